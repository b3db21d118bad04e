// GEMM for launches of a few hundred rows (gfx950):  Y = epilogue(X * W^T + bias), bf16 (units layout) or float32 (split layout) operands.
//
// Such a launch is bound by latency: a workgroup that streams its tile through the LDS spends most of every short K step
// on the barrier and the round trip of the loads.  Here nothing is staged and the K loop has no barrier: the four waves of a
// workgroup share the K range of one (32 NBI) x (32 NBJ) tile, each requests its MFMA operands straight into registers
// (both operand layouts are made of units a wave can load as they are, common.h), several steps ahead, and multiplies on its
// own.  The four partial tiles meet in the LDS once, at the end, where every thread adds up (wave 0 first) the eight
// consecutive features of one row that it then finishes and stores.  K may be split over blockIdx.y on top (float32 results).
#include "gemm_common.h"

namespace cubert {
namespace {

using namespace gemm_detail;

template <int ELT>
struct Operand;
// float32 split: a step is 16 k; per block of 32 rows three fragments, one per plane
template <>
struct Operand<kF32Split> {
    static constexpr int kFrags = 3, kStepK = 16;
    static __host__ __device__ size_t bytes(int rows, int K) { return split_bytes(rows, K); }
    static __device__ int lane_offset(int row0, int K, int l32, int g) { return (row0 >> 5) * (K / 16) * 3072 + (l32 + 32 * g) * 16; }
    static __device__ int block_stride(int K) { return K / 16 * 3072; }      // 32 rows further
    static constexpr int kStepBytes = 3072;
    static __device__ int frag_offset(int lane_off, int f) { return lane_off + f * 1024; }
};
// bf16 units: a step is 32 k (one 16 KiB block of 256 rows); per block of 32 rows two fragments, one per k-phase
template <>
struct Operand<kBF16> {
    static constexpr int kFrags = 2, kStepK = 32;
    static __host__ __device__ size_t bytes(int rows, int K) { return packed_bytes(rows, (size_t)K * 2); }
    static __device__ int lane_offset(int row0, int K, int l32, int g) {
        return (row0 >> 8) * (K / 32) * 16384 + (row0 & 255) * 64 + (l32 + 32 * g) * 16;
    }
    static __device__ int block_stride(int) { return 2048; }                 // 32 rows further in the same 256-row block
    static constexpr int kStepBytes = 16384;
    static __device__ int frag_offset(int lane_off, int f) { return lane_off + f * 1024; }
};

template <int ELT, int EPI, int NBI, int NBJ, int DEPTH>
__global__ __launch_bounds__(256, 2) void gemm_skinny_kernel(const GemmDev p) {
    typedef Operand<ELT> Op;
    constexpr int FR = Op::kFrags;
    constexpr bool QKV = EPI == kEpiQKV || EPI == kEpiQKVMap;
    constexpr bool F32OUT = EPI == kEpiBias || EPI == kEpiBiasRes;
    constexpr int ITEMS = NBI * NBJ / 2;                 // (row, eight features) pairs per thread at the end
    static_assert(NBI * NBJ % 2 == 0, "every thread finishes whole items");
    // [wave][block column of 32 features][row][128 bytes], 16-byte chunk c of row r in slot c ^ ((r >> 1) & 7)
    __shared__ __attribute__((aligned(16))) unsigned char part[4 * NBI * NBJ * 4096];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, g = lane >> 5;
    int tile_n, tile_m;
    tile_of_block<8>(blockIdx.x, p.tiles_n * p.tiles_m, p.tiles_n, p.xn_parts, &tile_n, &tile_m);
    const int n0 = tile_n * 32 * NBI, m0 = tile_m * 32 * NBJ;

    // steps of this wave: the wave-th quarter of the blockIdx.y-th share of K
    const int all = p.K / Op::kStepK;
    const int parts = 4 * p.splits, me = 4 * blockIdx.y + wave;
    const int s0 = (int)((long)all * me / parts), s1 = (int)((long)all * (me + 1) / parts);

    // rows past the operand (padded to 32 or 256 rows in memory) read as zero
    const __amdgpu_buffer_rsrc_t wres = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(p.W), 0, (int)Op::bytes(p.N, p.K), 0x00020000);
    const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(p.X), 0, (int)Op::bytes(p.M, p.K), 0x00020000);
    const int w_off = Op::lane_offset(n0, p.K, l32, g), x_off = Op::lane_offset(m0, p.K, l32, g), stride = Op::block_stride(p.K);
    u32x4_t wf[DEPTH][NBI][FR], xf[DEPTH][NBJ][FR];
    auto load = [&](int d, int step) {
        // Loads past the wave's share lie outside the descriptor (bit 31 of the lane offset): no traffic, zeros to multiply.
        // They are issued all the same: with a fixed number of loads per step the compiler waits for exactly the oldest ones.
        const int k = step * Op::kStepBytes, none = step < s1 ? 0 : (int)0x80000000u;
#pragma unroll
        for (int i = 0; i < NBI; ++i)
#pragma unroll
            for (int f = 0; f < FR; ++f)
                wf[d][i][f] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(wres, Op::frag_offset(w_off + i * stride, f) | none, k, 0));
#pragma unroll
        for (int j = 0; j < NBJ; ++j)
#pragma unroll
            for (int f = 0; f < FR; ++f)
                xf[d][j][f] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(xres, Op::frag_offset(x_off + j * stride, f) | none, k, 0));
    };
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
        load(d, s0 + d);
        __builtin_amdgcn_sched_barrier(0);
    }

    // what my items add at the end, requested now
    int row[ITEMS], c8[ITEMS];
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
        const int idx = tid + it * 256;
        if constexpr (EPI == kEpiBiasGelu) {       // units of 32 rows x 16 features
            const int unit = idx >> 6;
            row[it] = 32 * (unit / (2 * NBI)) + l32;
            c8[it] = 2 * (unit % (2 * NBI)) + g;
        } else {                                                       // row segments
            row[it] = idx / (4 * NBI);
            c8[it] = idx % (4 * NBI);
        }
    }
    f32x4_t bias[ITEMS][2], res[ITEMS][2];
    int tok[ITEMS];
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
        const int n = n0 + c8[it] * 8, m = m0 + row[it], mc = m < p.M ? m : p.M - 1;
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
            const int nc = n + 4 * hh < p.N ? n + 4 * hh : p.N - 4;
            bias[it][hh] = res[it][hh] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
            if (!F32OUT || blockIdx.y == 0) {                          // split K: bias and residual are added once
                bias[it][hh] = *reinterpret_cast<const f32x4_t*>(p.bias + nc);
                if constexpr (EPI == kEpiBiasRes) res[it][hh] = *reinterpret_cast<const f32x4_t*>(p.R + (size_t)mc * p.N + nc);
            }
        }
        tok[it] = mc;
        if constexpr (EPI == kEpiQKVMap) tok[it] = p.rowmap[mc];
    }

    f32x16_t acc[NBI][NBJ];
#pragma unroll
    for (int i = 0; i < NBI; ++i)
#pragma unroll
        for (int j = 0; j < NBJ; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
    auto multiply = [&](int d) {
        if constexpr (ELT == kBF16) {
#pragma unroll
            for (int f = 0; f < 2; ++f)
#pragma unroll
                for (int i = 0; i < NBI; ++i)
#pragma unroll
                    for (int j = 0; j < NBJ; ++j) mfma_chunk<kBF16>(wf[d][i][f], xf[d][j][f], acc[i][j]);
        } else {
            constexpr int wp[6] = {0, 0, 1, 1, 0, 2}, xp[6] = {0, 1, 0, 1, 2, 0};      // the plane products that count in float32
#pragma unroll
            for (int t = 0; t < 6; ++t)
#pragma unroll
                for (int i = 0; i < NBI; ++i)
#pragma unroll
                    for (int j = 0; j < NBJ; ++j) mfma_chunk<kBF16>(wf[d][i][wp[t]], xf[d][j][xp[t]], acc[i][j]);
        }
    };
    for (int s = s0; s < s1; s += DEPTH) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            multiply(d);
            load(d, s + d + DEPTH);
            __builtin_amdgcn_sched_barrier(0);       // left to itself the scheduler puts a round's loads together at its end
        }
    }

    unsigned char* mine = part + wave * (NBI * NBJ * 4096);
#pragma unroll
    for (int i = 0; i < NBI; ++i)
#pragma unroll
        for (int j = 0; j < NBJ; ++j)
#pragma unroll
            for (int qd = 0; qd < 4; ++qd) {
                const int r = 32 * j + l32;
                const f32x4_t v = {acc[i][j][4 * qd], acc[i][j][4 * qd + 1], acc[i][j][4 * qd + 2], acc[i][j][4 * qd + 3]};
                *reinterpret_cast<f32x4_t*>(mine + (i * NBJ * 32 + r) * 128 + (((2 * qd + g) ^ ((r >> 1) & 7)) << 4)) = v;
            }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
        const int r = row[it], m = m0 + r, n = n0 + c8[it] * 8;
        f32x4_t x[2];
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
            const int c = 2 * (c8[it] & 3) + hh;
            const unsigned char* src = part + ((c8[it] >> 2) * NBJ * 32 + r) * 128 + ((c ^ ((r >> 1) & 7)) << 4);
            x[hh] = *reinterpret_cast<const f32x4_t*>(src);
#pragma unroll
            for (int w = 1; w < 4; ++w) x[hh] += *reinterpret_cast<const f32x4_t*>(src + w * (NBI * NBJ * 4096));
            x[hh] += bias[it][hh];
            if constexpr (EPI == kEpiBiasRes) x[hh] += res[it][hh];
        }
        if constexpr (EPI == kEpiBiasGelu) {
#pragma unroll
            for (int hh = 0; hh < 2; ++hh)
#pragma unroll
                for (int e = 0; e < 4; ++e) x[hh][e] = ELT == kBF16 ? gelu_fast(x[hh][e]) : gelu_erf(x[hh][e]);
        }
        if (m >= p.M || n >= p.N) continue;                            // N % 8 == 0
        if constexpr (F32OUT) {
            float* dst = reinterpret_cast<float*>(p.Y) + ((size_t)blockIdx.y * p.M + m) * p.N + n;
            *reinterpret_cast<f32x4_t*>(dst) = x[0];
            *reinterpret_cast<f32x4_t*>(dst + 4) = x[1];
        } else {
            bf16x8_t pl[FR == 3 ? 3 : 1];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                if constexpr (ELT == kBF16) {
                    pl[0][e] = (__bf16)x[e >> 2][e & 3];
                } else {
                    __bf16 s0, s1, s2;
                    split_bf16x3(x[e >> 2][e & 3], s0, s1, s2);
                    pl[0][e] = s0; pl[1][e] = s1; pl[2][e] = s2;
                }
            }
            unsigned char* dst;
            if constexpr (QKV) {
                const int which = n >= 2 * p.hidden ? 2 : n >= p.hidden ? 1 : 0;
                const int hn = n - which * p.hidden, b = tok[it] / p.S, s = tok[it] - b * p.S;
                unsigned char* base = which == 2 ? p.vt : which ? p.k : p.q;
                if constexpr (ELT == kBF16) {
                    dst = base + ((((size_t)b * p.heads + (hn >> 6)) * p.S + s) * 64 + (hn & 63)) * 2;
                } else {
                    const int kk = (hn & 63) >> 4, half = (hn >> 3) & 1, pos = s & 31;
                    const size_t unit = ((((size_t)b * p.heads + (hn >> 6)) * (p.Sp >> 5) + (s >> 5)) * 4 + kk) * 3;
                    dst = base + unit * 1024 + half * 512 + (which == 2 ? attn_v_slot(pos, half, kk) : pos) * 16;
                }
            } else {
                dst = p.Y + (ELT == kBF16 ? units_offset(m, n * 2, p.N * 2 / 64) : split_offset(m, n, p.N));
            }
#pragma unroll
            for (int q = 0; q < (FR == 3 ? 3 : 1); ++q) *reinterpret_cast<bf16x8_t*>(dst + q * 1024) = pl[q];
        }
    }
}

template <int ELT, int NBI, int NBJ, int DEPTH>
bool launch_epi(const GemmDev& d, int epi, hipStream_t stream) {
    const dim3 grid(d.tiles_n * d.tiles_m, d.splits), block(256);
    switch (epi) {
        case kEpiBias: hipLaunchKernelGGL((gemm_skinny_kernel<ELT, kEpiBias, NBI, NBJ, DEPTH>), grid, block, 0, stream, d); break;
        case kEpiBiasGelu: hipLaunchKernelGGL((gemm_skinny_kernel<ELT, kEpiBiasGelu, NBI, NBJ, DEPTH>), grid, block, 0, stream, d); break;
        case kEpiQKV: hipLaunchKernelGGL((gemm_skinny_kernel<ELT, kEpiQKV, NBI, NBJ, DEPTH>), grid, block, 0, stream, d); break;
        case kEpiQKVMap: hipLaunchKernelGGL((gemm_skinny_kernel<ELT, kEpiQKVMap, NBI, NBJ, DEPTH>), grid, block, 0, stream, d); break;
        case kEpiBiasRes: hipLaunchKernelGGL((gemm_skinny_kernel<ELT, kEpiBiasRes, NBI, NBJ, DEPTH>), grid, block, 0, stream, d); break;
        default: set_error("gemm: unknown epilogue"); return false;
    }
    CUBERT_HIP_OK(hipGetLastError());
    return true;
}

}  // namespace

// elt kBF16 (both operands and a GELU result in the units layout; per-head row-major Q, K, V; float32 results) or kF32Split; tile kTileSkinny12 (32
// features x 64 tokens) or kTileSkinny22 (64 x 64); d.tiles_n / d.tiles_m for it; d.N % 8 == 0.
bool launch_gemm_skinny(const gemm_detail::GemmDev& d, int elt, int tile, int epilogue, hipStream_t stream) {
    const int step = elt == kBF16 ? 32 : 16;
    if (d.K % step != 0 || d.N % 8 != 0 || d.splits < 1 || 4 * d.splits > d.K / step) {
        set_error("gemm: the skinny kernel needs N a multiple of 8 and at least four K steps per split");
        return false;
    }
    if (elt == kBF16) {
        return tile == kTileSkinny12 ? launch_epi<kBF16, 1, 2, 6>(d, epilogue, stream) : launch_epi<kBF16, 2, 2, 4>(d, epilogue, stream);
    }
    return tile == kTileSkinny12 ? launch_epi<kF32Split, 1, 2, 4>(d, epilogue, stream) : launch_epi<kF32Split, 2, 2, 3>(d, epilogue, stream);
}

}  // namespace cubert
