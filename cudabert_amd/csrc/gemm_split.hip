// float32 GEMM on the bf16 matrix pipe (gfx950):  Y = epilogue(X * W^T + bias), X and W float32 in the split layout
// (common.h): three bf16 planes per operand, six plane products per float32 product, float32 accumulation.
//
// Same operand roles and epilogues as the other kernels (gemm.hip).  The K loops are hand-scheduled inline asm
// (gemm_split_128_loop.inc, gemm_split_256x128_loop.inc; pipeline and register plan in gen_gemm_asm.py).
//
// The 128 x 128 loop reads a step's fragments during the step before: 1024 x 768 x 768 (48 workgroups) 26.5 -> 23.8 us, 1024 x 3072 x
// 768 32.3 -> 30.6, 12800 x 1024 x 4096 513 -> 504; at 192 workgroups and more its loop runs at the rate the power limit allows.
//
// Bound: the matrix pipe at the socket's power limit.  9800 x 4096 x 1024 with GELU: 377 us, 218 TFLOP/s, i.e. 1.31 PFLOP/s of
// bf16 products; 25600 x 4096 x 1024 without it 1.43 at 1400 W of 1400 (a bf16 product of 8192^3 reaches 1.44 there: 0.97 pJ per
// operation both, where a bf16 FFN-in, whose fragments serve one product instead of two, spends 1.35), against 668 us, 123 TFLOP/s with the float32 MFMA, whose
// peak is 157; 19600 x 3072 x 1024: 535 us against 942.  Error against float64, root mean square of the result: 2.7e-7 at
// K = 1024 and 8.0e-7 at K = 4096, with the float32 MFMA 3.1e-7 and 9.1e-7 (fewer, larger accumulation steps).
#include "gemm_split_epilogue.h"

namespace cubert {
namespace {

using namespace gemm_detail;

#define CUBERT_V10(b) "v" #b "0", "v" #b "1", "v" #b "2", "v" #b "3", "v" #b "4", "v" #b "5", "v" #b "6", "v" #b "7", "v" #b "8", "v" #b "9"
#define CUBERT_ACC_22 [c00] "=&a"(acc[0][0]), [c01] "=&a"(acc[0][1]), [c10] "=&a"(acc[1][0]), [c11] "=&a"(acc[1][1])
#define CUBERT_ACC_42 CUBERT_ACC_22, [c20] "=&a"(acc[2][0]), [c21] "=&a"(acc[2][1]), [c30] "=&a"(acc[3][0]), [c31] "=&a"(acc[3][1])

// NBI x 2 accumulator blocks per wave: 2 for the 128 x 128 tile, 4 for the 256 features x 128 tokens one.
template <int EPI, int NBI>
__global__ __launch_bounds__(256, 2) void gemm_split_kernel(const GemmDev p) {
    constexpr int BN = 64 * NBI, BM = 128;
    constexpr int STAGES = NBI == 2 ? 3 : 2;
    constexpr int XOFF = 2 * NBI * 3072, STAGE = XOFF + 4 * 3072;      // W tile, then X tile of 16 k
    __shared__ __attribute__((aligned(1024))) unsigned char lds[STAGES * STAGE];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave >> 1, wm = wave & 1;
    const int l32 = lane & 31, g = lane >> 5;

    int tile_n, tile_m;
    tile_of_block<8>(blockIdx.x, p.tiles_n * p.tiles_m, p.tiles_n, p.xn_parts, &tile_n, &tile_m);
    const int n0 = tile_n * BN, m0 = tile_m * BM;

    // Descriptors that start at the tile's first row block, so that no operand size reaches 32 bits; row blocks past
    // the end read as zero.
    const int rb_stride = p.K / 16 * 3072;
    const unsigned long long wa = reinterpret_cast<unsigned long long>(p.W) + (unsigned long long)(n0 >> 5) * rb_stride;
    const unsigned long long xa = reinterpret_cast<unsigned long long>(p.X) + (unsigned long long)(m0 >> 5) * rb_stride;
    const int wleft = (p.N + 31) / 32 - (n0 >> 5), xleft = (p.M + 31) / 32 - (m0 >> 5);
    const u32x4_t wres = {(unsigned)wa, (unsigned)(wa >> 32) & 0xffffu, (unsigned)((wleft < BN / 32 ? wleft : BN / 32) * rb_stride), 0x00020000u};
    const u32x4_t xres = {(unsigned)xa, (unsigned)(xa >> 32) & 0xffffu, (unsigned)((xleft < BM / 32 ? xleft : BM / 32) * rb_stride), 0x00020000u};
    const int v0 = wave * rb_stride + lane * 16;
    const int rb4 = 4 * rb_stride;
    const int lds_base = (int)(size_t)(__attribute__((address_space(3))) unsigned char*)lds;
    const int wb = lds_base + wn * NBI * 3072 + lane * 16;
    const int xb = lds_base + wm * 2 * 3072 + lane * 16;               // + XOFF is in the read offsets
    const int m0b = __builtin_amdgcn_readfirstlane(lds_base + wave * 3072);
    // 16-k steps of this workgroup: all of K, or (split K) the blockIdx.y-th share of it
    const int ks = p.K / 16;
    const int s0 = (int)((long)ks * blockIdx.y / p.splits), s1 = (int)((long)ks * (blockIdx.y + 1) / p.splits);
    const int steps = s1 - s0, k0 = s0 * 3072, kmax = (s1 - 1) * 3072;

    f32x16_t acc[NBI][2];       // zeroed inside the asm block
    if constexpr (NBI == 2) {
        asm volatile(
#include "gemm_split_128_loop.inc"
            : CUBERT_ACC_22
            : [wb] "v"(wb), [xb] "v"(xb), [wv0] "v"(v0), [xv0] "v"(v0), [wres] "s"(wres), [xres] "s"(xres),
              [m0b] "s"(m0b), [k0] "s"(k0), [kmax] "s"(kmax), [steps] "s"(steps)
            : "memory", "scc", "m0", "s92", "s93", "s94", "s95", "s96", "s97", CUBERT_V10(4), CUBERT_V10(5), CUBERT_V10(6),
              CUBERT_V10(7), CUBERT_V10(8), CUBERT_V10(9), CUBERT_V10(10), CUBERT_V10(11), CUBERT_V10(12), CUBERT_V10(13), "v140",
              "v141", "v142", "v143", "v144", "v145");
    } else {
        asm volatile(
#include "gemm_split_256x128_loop.inc"
            : CUBERT_ACC_42
            : [wb] "v"(wb), [xb] "v"(xb), [wv0] "v"(v0), [xv0] "v"(v0), [wres] "s"(wres), [xres] "s"(xres), [rb4] "s"(rb4),
              [m0b] "s"(m0b), [k0] "s"(k0), [kmax] "s"(kmax), [steps] "s"(steps)
            : "memory", "scc", "m0", "s92", "s93", "s94", "s95", "s96", "s97", "v36", "v37", "v38", "v39", CUBERT_V10(4), CUBERT_V10(5),
              CUBERT_V10(6), CUBERT_V10(7), CUBERT_V10(8), CUBERT_V10(9), CUBERT_V10(10), CUBERT_V10(11), "v120");
    }

    // The block ends with all loads landed and a barrier: the whole LDS is free for staging.
    constexpr bool SPLITK = EPI == kEpiBias || EPI == kEpiBiasRes;
    f32x4_t bias[4 * NBI];
    const int nb = n0 + wn * 32 * NBI, mb = m0 + wm * 64;
    if constexpr (!gemm_bias_at_readout<kF32, EPI>()) gemm_load_bias<NBI, SPLITK>(p, nb, g, bias);
    if constexpr (EPI == kEpiBiasGelu || EPI == kEpiQKV || EPI == kEpiQKVMap)
        split_epilogue<EPI, NBI, 2>(p, acc, bias, nb, mb, l32, g);
    else
        gemm_epilogue<kF32, EPI, NBI, 2, SPLITK, 4, true>(p, acc, bias, nb, mb, l32, g, lds + wave * (NBI * 4096));
}

template <int NBI>
bool launch_epi(const GemmDev& d, int epi, hipStream_t stream) {
    const dim3 grid(d.tiles_n * d.tiles_m, d.splits), block(256);
    switch (epi) {
        case kEpiBias: hipLaunchKernelGGL((gemm_split_kernel<kEpiBias, NBI>), grid, block, 0, stream, d); break;
        case kEpiBiasGelu: hipLaunchKernelGGL((gemm_split_kernel<kEpiBiasGelu, NBI>), grid, block, 0, stream, d); break;
        case kEpiQKV: hipLaunchKernelGGL((gemm_split_kernel<kEpiQKV, NBI>), grid, block, 0, stream, d); break;
        case kEpiQKVMap: hipLaunchKernelGGL((gemm_split_kernel<kEpiQKVMap, NBI>), grid, block, 0, stream, d); break;
        case kEpiBiasRes: hipLaunchKernelGGL((gemm_split_kernel<kEpiBiasRes, NBI>), grid, block, 0, stream, d); break;
        default: set_error("gemm: unknown epilogue"); return false;
    }
    CUBERT_HIP_OK(hipGetLastError());
    return true;
}

}  // namespace

// d.tiles_n / d.tiles_m for the tile (128: 128 x 128, kTile256x128: 256 features x 128 tokens); d.K % 16 == 0,
// 1 <= d.splits <= d.K / 16.
bool launch_gemm_split(const gemm_detail::GemmDev& d, int tile, int epilogue, hipStream_t stream) {
    if (d.K % 16 != 0 || d.K < 16 || d.splits < 1 || d.splits > d.K / 16) {
        set_error("gemm: split operands need K to be a multiple of 16 and at most K / 16 splits");
        return false;
    }
    return tile == kTile256x128 ? launch_epi<4>(d, epilogue, stream) : launch_epi<2>(d, epilogue, stream);
}

}  // namespace cubert
