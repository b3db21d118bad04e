// float32 GEMM on split operands for launches of a few hundred to a few thousand rows (gfx950):  Y = epilogue(X * W^T + bias).
//
// The four waves of a workgroup share K: each multiplies its quarter of it for the whole tile, (32 NBI) features x 128 tokens, with
// operands that go straight from memory into registers (the split layout is made of MFMA operands, common.h).  No operand is staged
// and the K loop has no barrier; a wave has its SIMD and all of the registers to itself.  A step of 16 k of the 96 x 128 tile is 72 MFMAs, 2304 clocks,
// on 21 loads of 1 KiB, which go out between the MFMAs of the step before: 37 bytes a clock and CU of the 64 that its L2 gives.
// The partial tiles meet in the LDS once, at the end: wave w finishes token block w.  K may be split over workgroups on top (float32
// results).
//
// Against a tile staged in the LDS this takes a third of a workgroup's work per wave without its barriers, and a tile of 96 features makes one
// even round of launches that 128 x 128 leaves a quarter or half of the chip idle in: 1024 x 3072 x 768 256 workgroups instead of 192.
// Microseconds, weights from memory, LayerNorm included, against 128 x 128 with its best split:  1024 rows of BERT-base, QKV 28.7 -> 24.0,
// attn-out 23.2 -> 17.5, FFN-in 31.6 -> 28.3, FFN-out 39.1 -> 33.0; 512 rows of BERT-large, QKV 33.6 -> 23.9.
// Bound: 1.05 us a step of the 96 x 128 tile (0.96 at the peak rate of the matrix pipe), 0.9 of 64 x 128 and 0.7 of 32 x 128, which their fetches
// bound (80 to 90 GB/s a CU) where few CUs work; with all of them 1.3 to 1.5 us, the socket being at its power limit (1.6 PFLOP/s of bf16 products).
// Around the loop (time stamps, 1024 x 3072 x 768): 2.1 us until it begins, 1.1 for its first operands, 1.1 for the exchange, 2.6 for Q, K and V, 1.6
// for a float32 result, GELU 7.3 with the library's erff and some 4 with a polynomial of 24 issue slots a value (gelu_erf: 30); 3.6 between launches.  Without divisions on the device and with what
// addresses take in registers at the start, against tile_of_block and the argument record: passes of 270 to 2048 rows 1.1 to 2.4 % (8 lines of 128,
// BERT-base, 1665 -> 1626 us).
// Steps in flight beside the one at work: one; two are 2 % slower.
#include "gemm_split_epilogue.h"

namespace cubert {
namespace {

using namespace gemm_detail;

constexpr int kWaves = 4, kNBJ = 4, kDepth = 2;

constexpr int kGroupM = 8;

// What the operands' addresses take comes as arguments of its own, thirteen words that arrive in registers, with every division done by the host.
// Workgroup -> tile as in tile_of_block: xn (low byte of xn_shifts) = log2(xn_parts) + 1 or 0, cell = features' tiles << 16 | tokens' tiles of an XCD's cell (xn > 0) or of the
// grid, run = tiles / 8 << 3 | tiles % 8; divisors kGroupM * features' tiles of the cell and the bands of its last group, their shifts
// in the other bytes of xn_shifts.
// A wave has share >> 16 steps of 16 k, one more for the first share & 65535 of the kWaves * splits waves of a tile.
template <int EPI, int NBI>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(1, 1))) void gemm_split_share_kernel(
    const unsigned char* W, const unsigned char* X, int M, int N, int K, unsigned share_extra, int xn_shifts, unsigned cell, int run, unsigned group_magic,
    unsigned last_magic, const GemmDev p) {
    constexpr bool F32OUT = EPI == kEpiBias || EPI == kEpiBiasRes;
    // [token block][source wave ^ token block, less one][block of 32 features][quad][lane]
    __shared__ __attribute__((aligned(16))) unsigned char part[kNBJ * 3 * NBI * 4096];

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l32 = lane & 31, g = lane >> 5;
    const int xcd = blockIdx.x & 7, n_count = cell >> 16, m_count = cell & 65535, xn = xn_shifts & 255;
    int t = blockIdx.x >> 3, tile_n = 0, tile_m = 0;
    if (xn) {
        tile_n = (xcd & ((1 << (xn - 1)) - 1)) * n_count;
        tile_m = (xcd >> (xn - 1)) * m_count;
    } else {
        t += xcd * (run >> 3) + (xcd < (run & 7) ? xcd : run & 7);
    }
    const int group = div_by(t, group_magic, xn_shifts >> 8), r = t - group * kGroupM * n_count, bands = m_count - group * kGroupM;
    const int c = bands >= kGroupM ? r / kGroupM : div_by(r, last_magic, xn_shifts >> 16);
    tile_n += c;
    tile_m += group * kGroupM + r - c * (bands >= kGroupM ? kGroupM : bands);
    const int n0 = tile_n * 32 * NBI, m0 = tile_m * 32 * kNBJ;

    const int split = blockIdx.y, me = kWaves * split + wave, share = share_extra >> 16, extra = share_extra & 65535;
    const int s0 = me * share + (me < extra ? me : extra), s1 = s0 + share + (me < extra ? 1 : 0);

    // descriptors that start at the tile's first row block, so that no operand size reaches 32 bits; row blocks past the end read as zero
    const int rb_stride = K / 16 * 3072;
    const int wleft = (N + 31) / 32 - (n0 >> 5), xleft = (M + 31) / 32 - (m0 >> 5);
    const __amdgpu_buffer_rsrc_t wres = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<unsigned char*>(W) + (size_t)(n0 >> 5) * rb_stride, 0, (wleft < NBI ? wleft : NBI) * rb_stride, 0x00020000);
    const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<unsigned char*>(X) + (size_t)(m0 >> 5) * rb_stride, 0, (xleft < kNBJ ? xleft : kNBJ) * rb_stride, 0x00020000);

    int off[kNBJ];                                                     // of my 16 bytes in each row block (NBI <= kNBJ)
#pragma unroll
    for (int j = 0; j < kNBJ; ++j) off[j] = j * rb_stride + lane * 16;
    u32x4_t wf[kDepth][3][NBI], xf[kDepth][3][kNBJ];
    // Loads past the wave's share lie outside the descriptor (bit 31 of the lane offset): no traffic.  They are issued all the same: with a
    // fixed number of loads in flight the compiler waits for exactly the oldest ones.
    auto load = [&](int d, int step) {
        const int k = step * 3072, none = step < s1 ? 0 : (int)0x80000000u;
#pragma unroll
        for (int pl = 0; pl < 3; ++pl) {
#pragma unroll
            for (int i = 0; i < NBI; ++i)
                wf[d][pl][i] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(wres, (off[i] | none) + pl * 1024, k, 0));
#pragma unroll
            for (int j = 0; j < kNBJ; ++j)
                xf[d][pl][j] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(xres, (off[j] | none) + pl * 1024, k, 0));
        }
    };
    f32x16_t acc[NBI][kNBJ];
#pragma unroll
    for (int i = 0; i < NBI; ++i)
#pragma unroll
        for (int j = 0; j < kNBJ; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
    auto multiply = [&](int d) {
        constexpr int wp[6] = {0, 0, 1, 1, 0, 2}, xp[6] = {0, 1, 0, 1, 2, 0};      // the plane products that count in float32
#pragma unroll
        for (int t = 0; t < 6; ++t)
#pragma unroll
            for (int i = 0; i < NBI; ++i)
#pragma unroll
                for (int j = 0; j < kNBJ; ++j) mfma_chunk<kBF16>(wf[d][wp[t]][i], xf[d][xp[t]][j], acc[i][j]);
    };
    // a step's loads are spread over its MFMAs
    auto interleave = [] {
#pragma unroll
        for (int n = 0; n < 3 * (NBI + kNBJ); ++n) {
            __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 6 * NBI * kNBJ / (3 * (NBI + kNBJ)), 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int d = 0; d < kDepth - 1; ++d) {
        load(d, s0 + d);
        __builtin_amdgcn_sched_barrier(0);
    }
    int s = s0;
    for (; s + kDepth <= s1; s += kDepth) {
#pragma unroll
        for (int d = 0; d < kDepth; ++d) {
            load((d + kDepth - 1) % kDepth, s + d + kDepth - 1);
            multiply(d);
            interleave();
        }
    }

    // what the results take, requested behind the last steps
    const int mb = m0 + 32 * wave;
    constexpr int SEG = F32OUT ? NBI : 1;
    f32x4_t bias[F32OUT ? NBI : 4 * NBI], res[SEG][4];
    if constexpr (F32OUT) {
#pragma unroll
        for (int i = 0; i < NBI; ++i) {
            const int n = n0 + 32 * i + 4 * (lane & 7), nc = n < p.N ? n : p.N - 4;
            bias[i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
            if (split == 0) bias[i] = *reinterpret_cast<const f32x4_t*>(p.bias + nc);          // split K: bias and residual are added once
#pragma unroll
            for (int it = 0; it < 4; ++it) {
                const int m = mb + 8 * it + (lane >> 3), mc = m < p.M ? m : p.M - 1;
                res[i][it] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
                if constexpr (EPI == kEpiBiasRes)
                    if (split == 0) res[i][it] = *reinterpret_cast<const f32x4_t*>(p.R + (size_t)mc * p.N + nc);
            }
        }
    } else {
        gemm_load_bias<NBI>(p, n0, g, bias);
    }
#pragma unroll
    for (int d = 0; d < kDepth - 1; ++d)
        if (s + d < s1) multiply(d);

    f32x16_t own[NBI][1];
#pragma unroll
    for (int j = 0; j < kNBJ; ++j) {
        if (j == wave) {
#pragma unroll
            for (int i = 0; i < NBI; ++i) own[i][0] = acc[i][j];
        } else {
            unsigned char* dst = part + (j * 3 + (wave ^ j) - 1) * NBI * 4096 + lane * 16;
#pragma unroll
            for (int i = 0; i < NBI; ++i)
#pragma unroll
                for (int qd = 0; qd < 4; ++qd)
                    *reinterpret_cast<f32x4_t*>(dst + i * 4096 + qd * 1024) =
                        f32x4_t{acc[i][j][4 * qd], acc[i][j][4 * qd + 1], acc[i][j][4 * qd + 2], acc[i][j][4 * qd + 3]};
        }
    }
    __syncthreads();
    // (wave 0 + wave 1) + (wave 2 + wave 3), whichever of them this is
    unsigned char* mine = part + wave * 3 * NBI * 4096;
#pragma unroll
    for (int i = 0; i < NBI; ++i)
#pragma unroll
        for (int qd = 0; qd < 4; ++qd) {
            const unsigned char* src = mine + i * 4096 + qd * 1024 + lane * 16;
            const f32x4_t a = *reinterpret_cast<const f32x4_t*>(src), b = *reinterpret_cast<const f32x4_t*>(src + NBI * 4096),
                          c = *reinterpret_cast<const f32x4_t*>(src + 2 * NBI * 4096);
#pragma unroll
            for (int e = 0; e < 4; ++e) own[i][0][4 * qd + e] = (own[i][0][4 * qd + e] + a[e]) + (b[e] + c[e]);
        }
    if constexpr (!F32OUT) {
        split_epilogue<EPI, NBI, 1>(p, own, bias, n0, mb, l32, g);
    } else {
        // through the LDS (the wave's own part of it, read out by now), so that they leave as row segments of 128 bytes: chunk c of row r
        // in slot c ^ ((r >> 1) & 7)
#pragma unroll
        for (int i = 0; i < NBI; ++i) {
            unsigned char* buf = mine + i * 4096;
#pragma unroll
            for (int qd = 0; qd < 4; ++qd)
                *reinterpret_cast<f32x4_t*>(buf + l32 * 128 + (((2 * qd + g) ^ ((l32 >> 1) & 7)) << 4)) =
                    f32x4_t{own[i][0][4 * qd], own[i][0][4 * qd + 1], own[i][0][4 * qd + 2], own[i][0][4 * qd + 3]};
#pragma unroll
            for (int it = 0; it < 4; ++it) {
                const int r = 8 * it + (lane >> 3), m = mb + r, n = n0 + 32 * i + 4 * (lane & 7);
                f32x4_t x = *reinterpret_cast<const f32x4_t*>(buf + r * 128 + (((lane & 7) ^ ((r >> 1) & 7)) << 4));
                x += bias[i];
                if constexpr (EPI == kEpiBiasRes) x += res[i][it];
                if (m < p.M && n < p.N) *reinterpret_cast<f32x4_t*>(reinterpret_cast<float*>(p.Y) + ((size_t)split * p.M + m) * p.N + n) = x;
            }
        }
    }
}

template <int NBI>
bool launch_epi(const GemmDev& d, int epi, hipStream_t stream) {
    const dim3 grid(d.tiles_n * d.tiles_m, d.splits), block(64 * kWaves);
    const int total = d.tiles_n * d.tiles_m, steps = d.K / 16, waves = kWaves * d.splits;
    int xn = d.xn_parts == 4 ? 3 : d.xn_parts == 2 ? 2 : 0;
    if (xn && (total % 8 != 0 || d.tiles_n % d.xn_parts != 0 || d.tiles_m % (8 / d.xn_parts) != 0)) xn = 0;
    const int n_count = xn ? d.tiles_n / d.xn_parts : d.tiles_n, m_count = xn ? d.tiles_m / (8 / d.xn_parts) : d.tiles_m;
    if (n_count > 65535 || m_count > 65535 || steps / waves > 65535 || (long)d.tiles_n * d.tiles_m >= 1L << 24) { set_error("gemm: too many tiles"); return false; }
    const unsigned share = (unsigned)(steps / waves) << 16 | steps % waves, cell = (unsigned)n_count << 16 | m_count;
    const Divisor group = divisor_of(kGroupM * n_count), last = divisor_of(m_count % kGroupM);
    const int xn_shifts = xn | group.shift << 8 | last.shift << 16;
#define CUBERT_SHARE(E) hipLaunchKernelGGL((gemm_split_share_kernel<E, NBI>), grid, block, 0, stream, d.W, d.X, d.M, d.N, d.K, share, xn_shifts, cell, \
                                           total / 8 << 3 | total % 8, group.magic, last.magic, d)
    switch (epi) {
        case kEpiBias: CUBERT_SHARE(kEpiBias); break;
        case kEpiBiasGelu: CUBERT_SHARE(kEpiBiasGelu); break;
        case kEpiQKV: CUBERT_SHARE(kEpiQKV); break;
        case kEpiQKVMap: CUBERT_SHARE(kEpiQKVMap); break;
        case kEpiBiasRes: CUBERT_SHARE(kEpiBiasRes); break;
        default: set_error("gemm: unknown epilogue"); return false;
    }
#undef CUBERT_SHARE
    CUBERT_HIP_OK(hipGetLastError());
    return true;
}

}  // namespace

// d.tiles_n / d.tiles_m for the tile (share_features(tile) x 128 tokens); d.K % 16 == 0, a K step at least for each of the 4 splits waves.
bool launch_gemm_split_share(const gemm_detail::GemmDev& d, int tile, int epilogue, hipStream_t stream) {
    if (d.K % 16 != 0 || d.splits < 1 || 4 * d.splits > d.K / 16) {
        set_error("gemm: the tiles whose waves share K need K to be a multiple of 16 and four K steps per split");
        return false;
    }
    switch (share_features(tile)) {
        case 32: return launch_epi<1>(d, epilogue, stream);
        case 64: return launch_epi<2>(d, epilogue, stream);
        default: return launch_epi<3>(d, epilogue, stream);
    }
}

}  // namespace cubert
