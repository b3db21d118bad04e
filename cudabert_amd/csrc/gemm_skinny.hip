// GEMM for launches of a few hundred rows (gfx950):  Y = epilogue(X * W^T + bias), bf16 (units layout) or float32 (split layout) operands.
//
// Such a launch is bound by latency: a workgroup that streams its tile through the LDS spends most of every short K step
// on the barrier and the round trip of the loads.  Here nothing is staged and the K loop has no barrier: the eight waves of a
// workgroup share the K range of one (32 NBI) x (32 NBJ) tile, each requests its MFMA operands straight into registers
// (both operand layouts are made of units a wave can load as they are, common.h), several steps ahead, and multiplies on its
// own.  The partial tiles meet in the LDS once, at the end, where every thread adds up the four consecutive features of one row
// that it then finishes and stores.  K may be split over workgroups on top (float32 results).
//
// What such a launch lasts (time stamps, bf16, 17 x 4096 x 1024, weights in the L2): 0.1 us until a wave runs, 0.55 until it has
// addresses where the kernel divides (the workgroup's number by tiles, the wave's by parts), 1.3 until operands arrive, a CU taking 64 bytes a
// clock (148 GB/s) from its L2; 0.3 for products, 0.2 for the exchange, 0.65 for results where 128 threads finish eight features each, and
// 1.3 between launches.  Weights that are not in the L2: 2.3 more in bf16, 5 with split operands.  Hence no division on the device, four
// features a thread, and eight waves with the whole of a K of 1024 in flight.  With four waves, eight features and divisions -> now, weights
// from memory, smallest tile that gives each CU one workgroup: bf16 17 x 2304 x 768 4.8 -> 3.6 us, 17 x 4096 x 1024 7.8 -> 5.5, 128 x 3072 x 768
// 5.5 -> 4.6, 128 x 4096 x 1024 7.9 -> 6.4; split operands 17 x 4096 x 1024 11.4 -> 10.3, 64 x 3072 x 1024 13.1 -> 9.8.
#include "gemm_skinny_map.h"

namespace cubert {
namespace {

using namespace gemm_detail;

// (An operand is smaller than 2 GiB, so that its size and offsets in it take 32 bits: the size by 64 bits was a dozen instructions of a wave's way to
// its first load.)
template <int ELT>
struct Operand;
// float32 split: a step is 16 k; per block of 32 rows three fragments, one per plane
template <>
struct Operand<kF32Split> {
    static constexpr int kFrags = 3, kStepK = 16;
    static __device__ unsigned bytes(int rows, int K) { return ((unsigned)(rows + 31) >> 5) * (K >> 4) * 3072; }      // split_bytes
    static __device__ int lane_offset(int row0, int K, int l32, int g) { return (row0 >> 5) * (K >> 4) * 3072 + (l32 + 32 * g) * 16; }
    static __device__ int block_stride(int K) { return (K >> 4) * 3072; }    // 32 rows further
    static constexpr int kStepBytes = 3072;
    static __device__ int frag_offset(int lane_off, int f) { return lane_off + f * 1024; }
};
// bf16 units: a step is 32 k (one 16 KiB block of 256 rows); per block of 32 rows two fragments, one per k-phase
template <>
struct Operand<kBF16> {
    static constexpr int kFrags = 2, kStepK = 32;
    static __device__ unsigned bytes(int rows, int K) { return ((unsigned)(rows + 255) >> 8) * (K >> 5) * 16384; }    // packed_bytes
    static __device__ int lane_offset(int row0, int K, int l32, int g) {
        return (row0 >> 8) * (K >> 5) * 16384 + (row0 & 255) * 64 + (l32 + 32 * g) * 16;
    }
    static __device__ int block_stride(int) { return 2048; }                 // 32 rows further in the same 256-row block
    static constexpr int kStepBytes = 16384;
    static __device__ int frag_offset(int lane_off, int f) { return lane_off + f * 1024; }
};

constexpr int kWaves = 8;

// What the kernel needs of a GemmDev, with every division done by the host.  What the operands' addresses take comes as arguments of
// its own, fourteen words that arrive in registers; the rest, loaded, is needed when the operands are under way.
struct SkinnyRest {
    const float *bias, *R;
    unsigned char *Y, *k, *vt;          // QKV: Y is q
    const int* rowmap;
    int S, Sp, heads;
    unsigned s_magic, s_shift;          // divisor S
    int v_rowmajor;                     // bf16 QKV: V like k; else [B, heads, 64, Sp]
};

// Workgroup -> tile and part of K: skinny_tile (gemm_skinny_map.h).  A wave has `share` K steps, one more for the first `extra` of the
// kWaves * splits waves of a tile.
template <int ELT, int EPI, int NBI, int NBJ, int DEPTH>
__global__ __launch_bounds__(64 * kWaves, 2) void gemm_skinny_kernel(const unsigned char* W, const unsigned char* X, int M, int N, int K,
                                                                     int per_xcd, int tiles_m, unsigned m_magic, unsigned split_magic,
                                                                     int splits_more, unsigned shifts, int share_extra, const SkinnyRest p) {
    typedef Operand<ELT> Op;
    constexpr int FR = Op::kFrags, THREADS = 64 * kWaves;
    constexpr bool QKV = EPI == kEpiQKV || EPI == kEpiQKVMap;
    constexpr bool F32OUT = EPI == kEpiBias || EPI == kEpiBiasRes;
    // the result leaves in units of 32 rows x 16 features, or in row segments
    constexpr bool UNITS = EPI == kEpiBiasGelu || (QKV && ELT == kF32Split);
    constexpr int ALL = 256 * NBI * NBJ, ITEMS = (ALL + THREADS - 1) / THREADS;      // (row, four features) pairs: all, and per thread
    // [wave][block column of 32 features][row][128 bytes], 16-byte chunk c of row r in slot c ^ ((r >> 1) & 7)
    constexpr int PART = NBI * NBJ * 4096;
    __shared__ __attribute__((aligned(16))) unsigned char part[kWaves * PART];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, g = lane >> 5;
    const int share = share_extra >> 11, extra = share_extra & 2047;
    int tile_n, tile_m, split;
    if (!skinny_tile(blockIdx.x, blockIdx.y, (int)((unsigned)(N + 32 * NBI - 1) / (32 * NBI)), per_xcd, tiles_m, m_magic, split_magic, splits_more, shifts, &tile_n, &tile_m, &split))
        return;                                                        // the whole workgroup: no barrier has been met
    const int n0 = tile_n * 32 * NBI, m0 = tile_m * 32 * NBJ;

    const int me = kWaves * split + wave;
    const int s0 = me * share + (me < extra ? me : extra), s1 = s0 + share + (me < extra ? 1 : 0);

    // rows past the operand (padded to 32 or 256 rows in memory) read as zero
    const __amdgpu_buffer_rsrc_t wres = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(W), 0, (int)Op::bytes(N, K), 0x00020000);
    const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(X), 0, (int)Op::bytes(M, K), 0x00020000);
    const int w_off = Op::lane_offset(n0, K, l32, g), x_off = Op::lane_offset(m0, K, l32, g), stride = Op::block_stride(K);
    u32x4_t wf[DEPTH][NBI][FR], xf[DEPTH][NBJ][FR];
    auto load = [&](int d, int step) {
        // Loads past the wave's share lie outside the descriptor (bit 31 of the lane offset): nothing is fetched, but the CU takes as long
        // over their addresses as over others', hence the depths (launch_depth).
        // They are issued all the same: with a fixed number of loads in flight the compiler waits for exactly the oldest ones.
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

    // what my items add at the end, requested now, and where they go
    int row[ITEMS], c4[ITEMS];
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
        const int idx = (tid + it * THREADS) % ALL;                    // (threads past the last item repeat one and do not store it)
        if constexpr (UNITS) {                                         // half unit by half unit, 512 bytes each
            const int unit = idx >> 7;
            row[it] = 32 * (unit / (2 * NBI)) + ((idx >> 1) & 31);
            c4[it] = 4 * (unit % (2 * NBI)) + 2 * ((idx >> 6) & 1) + (idx & 1);
        } else {
            row[it] = idx / (8 * NBI);
            c4[it] = idx % (8 * NBI);
        }
    }
    f32x4_t bias[ITEMS], res[ITEMS];
    int tok[ITEMS];
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
        const int n = n0 + c4[it] * 4, m = m0 + row[it], mc = m < M ? m : M - 1, nc = n < N ? n : N - 4;
        bias[it] = res[it] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
        if (!F32OUT || split == 0) {                                   // split K: bias and residual are added once
            bias[it] = *reinterpret_cast<const f32x4_t*>(p.bias + nc);
            if constexpr (EPI == kEpiBiasRes) res[it] = *reinterpret_cast<const f32x4_t*>(p.R + (size_t)mc * N + nc);
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
    int s = s0;
    for (; s + DEPTH < s1; s += DEPTH) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            multiply(d);
            load(d, s + d + DEPTH);
            __builtin_amdgcn_sched_barrier(0);       // left to itself the scheduler puts a round's loads together at its end
        }
    }
#pragma unroll
    for (int d = 0; d < DEPTH; ++d)
        if (s + d < s1) multiply(d);

    unsigned char* mine = part + wave * PART;
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
        const int r = row[it], m = m0 + r, n = n0 + c4[it] * 4;
        const unsigned char* src = part + ((c4[it] >> 3) * NBJ * 32 + r) * 128 + (((c4[it] & 7) ^ ((r >> 1) & 7)) << 4);
        f32x4_t p8[kWaves];
#pragma unroll
        for (int w = 0; w < kWaves; ++w) p8[w] = *reinterpret_cast<const f32x4_t*>(src + w * PART);
        f32x4_t x = ((p8[0] + p8[1]) + (p8[2] + p8[3])) + ((p8[4] + p8[5]) + (p8[6] + p8[7]));
        x += bias[it];
        if constexpr (EPI == kEpiBiasRes) x += res[it];
        if constexpr (EPI == kEpiBiasGelu) {
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = ELT == kBF16 ? gelu_fast(x[e]) : gelu_erf(x[e]);
        }
        if (m >= M || n >= N || (ALL < THREADS && tid >= ALL)) continue;
        if constexpr (F32OUT) {
            *reinterpret_cast<f32x4_t*>(reinterpret_cast<float*>(p.Y) + ((size_t)split * M + m) * N + n) = x;
        } else {
            bf16x4_t pl[FR == 3 ? 3 : 1];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if constexpr (ELT == kBF16) {
                    pl[0][e] = (__bf16)x[e];
                } else {
                    __bf16 a0, a1, a2;
                    split_bf16x3(x[e], a0, a1, a2);
                    pl[0][e] = a0; pl[1][e] = a1; pl[2][e] = a2;
                }
            }
            unsigned char* dst;
            if constexpr (QKV) {
                const int hidden = p.heads * 64;                       // a tile lies in one head: hidden and n0 are multiples of its width
                const int which = n0 >= 2 * hidden ? 2 : n0 >= hidden ? 1 : 0, head = (n0 - which * hidden) >> 6;
                const int hn = n & 63, b = div_by(tok[it], p.s_magic, p.s_shift), s = tok[it] - b * p.S;
                unsigned char* base = which == 2 ? p.vt : which ? p.k : p.Y;
                if constexpr (ELT == kBF16) {
                    if (which == 2 && !p.v_rowmajor) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) *reinterpret_cast<__bf16*>(base + ((((size_t)b * p.heads + head) * 64 + hn + e) * p.Sp + s) * 2) = pl[0][e];
                        continue;
                    }
                    dst = base + ((((size_t)b * p.heads + head) * p.S + s) * 64 + hn) * 2;
                } else {
                    const int kk = hn >> 4, half = (hn >> 3) & 1, pos = s & 31;
                    const size_t unit = ((((size_t)b * p.heads + head) * (p.Sp >> 5) + (s >> 5)) * 4 + kk) * 3;
                    dst = base + unit * 1024 + half * 512 + (which == 2 ? attn_v_slot(pos, half, kk) : pos) * 16 + (hn & 4) * 2;
                }
            } else {
                dst = p.Y + (ELT == kBF16 ? units_offset(m, n * 2, N * 2 / 64) : split_offset(m, n, N));
            }
#pragma unroll
            for (int q = 0; q < (FR == 3 ? 3 : 1); ++q) *reinterpret_cast<bf16x4_t*>(dst + q * 1024) = pl[q];
        }
    }
}

template <int ELT, int NBI, int NBJ, int DEPTH>
bool launch_epi(const GemmDev& d, int epi, hipStream_t stream) {
    SkinnyRest p{};
    p.bias = d.bias; p.R = d.R;
    p.Y = epi == kEpiQKV || epi == kEpiQKVMap ? d.q : d.Y;
    p.k = d.k; p.vt = d.vt; p.rowmap = d.rowmap;
    p.S = d.S; p.Sp = d.Sp; p.heads = d.heads;
    const Divisor by_s = divisor_of(d.S);
    p.s_magic = by_s.magic; p.s_shift = by_s.shift;
    p.v_rowmajor = d.v_rowmajor;
    SkinnyMap map;
    if (!skinny_map((d.N + 32 * NBI - 1) / (32 * NBI), (d.M + 32 * NBJ - 1) / (32 * NBJ), d.splits, d.xn_parts, &map)) { set_error("gemm: too many tiles"); return false; }
    const int waves = kWaves * d.splits, steps = d.K / Operand<ELT>::kStepK, share_extra = steps / waves << 11 | steps % waves;      // (splits < 256)
    const dim3 grid(map.grid_x, map.grid_y), block(64 * kWaves);
#define CUBERT_SKINNY(E) hipLaunchKernelGGL((gemm_skinny_kernel<ELT, E, NBI, NBJ, DEPTH>), grid, block, 0, stream, d.W, d.X, d.M, d.N, d.K, \
                                            map.per_xcd, map.tiles_m, map.m_magic, map.split_magic, map.splits_more, map.shifts, share_extra, p)
    switch (epi) {
        case kEpiBias: CUBERT_SKINNY(kEpiBias); break;
        case kEpiBiasGelu: CUBERT_SKINNY(kEpiBiasGelu); break;
        case kEpiQKV: CUBERT_SKINNY(kEpiQKV); break;
        case kEpiQKVMap: CUBERT_SKINNY(kEpiQKVMap); break;
        case kEpiBiasRes: CUBERT_SKINNY(kEpiBiasRes); break;
        default: set_error("gemm: unknown epilogue"); return false;
    }
#undef CUBERT_SKINNY
    CUBERT_HIP_OK(hipGetLastError());
    return true;
}

// Steps in flight: the fewest of the depths that hold a wave's share, or the last, as many as its 256 registers hold.  With the last for every
// share, most loads of narrow models were past it: six layers, us, last depth / chosen, hidden 64, float32, 17 rows 206 / 157, 2048 rows 270 / 222;
// hidden 128 17 rows 213 / 167, bf16 152 / 143; hidden 768 17 rows 253 / 226, bf16 168 / 163; level where a share fills it (hidden 1024, bf16 228 / 228).
template <int ELT, int NBI, int NBJ, int DEPTH, int... MORE>
bool launch_depth(const GemmDev& d, int share, int epi, hipStream_t stream) {
    if constexpr (sizeof...(MORE) > 0)
        if (share > DEPTH) return launch_depth<ELT, NBI, NBJ, MORE...>(d, share, epi, stream);
    return launch_epi<ELT, NBI, NBJ, DEPTH>(d, epi, stream);
}

}  // namespace

// elt kBF16 (both operands and a GELU result in the units layout; per-head Q, K, V; float32 results) or kF32Split; tile a
// skinny one; d.N % 8 == 0; d.xn_parts 0, 2 or 4 (skinny_map's cells).
bool launch_gemm_skinny(const gemm_detail::GemmDev& d, int elt, int tile, int epilogue, hipStream_t stream) {
    const int step = elt == kBF16 ? 32 : 16;
    if (d.K % step != 0 || d.N % 8 != 0 || d.splits < 1 || d.splits > 255 || 4 * d.splits > d.K / step) {
        set_error("gemm: the skinny kernel needs N a multiple of 8 and at least four K steps per split");
        return false;
    }
    const int share = (d.K / step + kWaves * d.splits - 1) / (kWaves * d.splits);
    if (elt == kBF16) {
        switch (tile) {
            case kTileSkinny11: return launch_depth<kBF16, 1, 1, 1, 2, 3, 4>(d, share, epilogue, stream);
            case kTileSkinny21: return launch_depth<kBF16, 2, 1, 1, 2, 3, 4>(d, share, epilogue, stream);
            case kTileSkinny12: return launch_depth<kBF16, 1, 2, 1, 2, 3, 4>(d, share, epilogue, stream);
            default: return launch_depth<kBF16, 2, 2, 1, 2, 3, 4>(d, share, epilogue, stream);
        }
    }
    switch (tile) {
        case kTileSkinny11: return launch_depth<kF32Split, 1, 1, 2, 4, 6, 8>(d, share, epilogue, stream);
        case kTileSkinny21: return launch_depth<kF32Split, 2, 1, 1, 2, 3, 5>(d, share, epilogue, stream);
        case kTileSkinny12: return launch_depth<kF32Split, 1, 2, 1, 2, 3, 5>(d, share, epilogue, stream);
        default: return launch_depth<kF32Split, 2, 2, 1, 2, 3>(d, share, epilogue, stream);
    }
}

}  // namespace cubert
