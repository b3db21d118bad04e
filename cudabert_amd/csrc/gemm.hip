// MFMA GEMM for gfx950 (MI355X):  Y = epilogue(X * W^T + bias).
//
// Both operands are K-contiguous ([rows, K]); a workgroup of four wave64s
// computes a BT x BT macro tile (BT features x BT tokens), each wave a
// (BT/2) x (BT/2) quadrant built from 32x32 MFMA blocks.  Per K step a slab of
// 128 bytes per row (64 bf16 / 32 f32) of both operands is loaded straight
// from global memory into LDS (buffer_load ... lds, one barrier per step): two
// LDS stages for the 256 and 128 tiles, four for the 64 tile, whose steps are so
// short that a single step of prefetch leaves every step waiting a full memory
// latency.
//
// LDS image of an operand tile: two sub-blocks (the two 64-byte halves of the
// K slab), each BT rows x 64 bytes; a row is four 16-byte chunks and chunk c
// of row r sits in slot c ^ ((r >> 2) & 3) (packed_swizzle), which spreads the
// 16-byte fragment reads of 8 or 16 consecutive rows over all banks.  This is
// also the on-device "packed" operand layout (common.h): a packed operand is
// stored as 16 KiB blocks of 256 rows x 64 bytes that already are this image,
// so loading a tile is a plain contiguous copy; an unpacked (row-major)
// operand is gathered into the same image by choosing which chunk each lane
// fetches.
//
// The weight tile feeds the MFMA "A" operand and the activation tile the "B"
// operand, i.e. the hardware computes Y^T blocks: a lane then owns one token
// and four consecutive output features per accumulator quad, which makes the
// row-major stores 8/16-byte vectors and lets the QKV epilogue write per-head
// layouts directly.
//
// The k index inside one MFMA is only a label: lane (row, g = lane / 32) feeds
// the 16-byte chunk 2*kk + g of its row for both operands, so A and B always
// pair identical k.  For f32 each chunk holds four k values consumed by four
// 32x32x2 MFMAs; for bf16 it holds eight consumed by one 32x32x16 MFMA.
//
// The 256 tile in bf16 has a hand-scheduled twin (gemm_bf16_256.hip); this
// file is the general kernel (any tile, f32, odd step counts).
#include <algorithm>
#include <cmath>

#include "gemm_common.h"

namespace cubert {

bool launch_gemm_bf16_t256(const gemm_detail::GemmDev& d, int out_elt, int epilogue, hipStream_t stream);
bool launch_gemm_bf16_t256x128(const gemm_detail::GemmDev& d, int out_elt, int epilogue, hipStream_t stream);
bool launch_gemm_bf16_t128(const gemm_detail::GemmDev& d, int out_elt, int epilogue, hipStream_t stream);
bool launch_gemm_bf16_t256x128_deep(const gemm_detail::GemmDev& d, int out_elt, int epilogue, hipStream_t stream);
bool launch_gemm_bf16_t256x192_ln(const gemm_detail::GemmDev& d, hipStream_t stream);
bool launch_gemm_skinny(const gemm_detail::GemmDev& d, int elt, int tile, int epilogue, hipStream_t stream);
bool launch_gemm_split_share(const gemm_detail::GemmDev& d, int tile, int epilogue, hipStream_t stream);
bool launch_gemm_split(const gemm_detail::GemmDev& d, int tile, int epilogue, hipStream_t stream);
int gemm_pick_tile(int M, int N, int K, int elt);

namespace {

using namespace gemm_detail;

template <int ELT, int OUT, int EPI, int BT, int NS>
__global__ __launch_bounds__(256) void gemm_kernel(const GemmDev p) {
    constexpr int ES = (ELT == kBF16) ? 2 : 4;       // operand element size
    constexpr int NB = BT / 64;                      // 32x32 blocks per wave and dimension
    constexpr int GROUPS = BT / 32;                  // loads each wave issues per operand tile and step
    constexpr int SUB = BT * 64;                     // one sub-block (64-byte half of the K slab)
    constexpr int TILE_BYTES = 2 * SUB;              // one operand tile in LDS
    constexpr int SBDIV = BT / 16;                   // 16-row groups per sub-block
    constexpr int BK = 128 / ES;                     // K elements per step

    // NS = LDS stages: two, or four for the 64 tile of a launch with few workgroups (64 KiB; with
    // many workgroups the four resident ones that two stages allow hide the latency better).
    static_assert(NS == 2 || (NS == 4 && BT == 64), "four stages only fit the 64 tile");
    constexpr int LPT = 2 * GROUPS;                  // loads a wave issues per step
    // s_waitcnt vmcnt(n) with n = the loads of the NS - 2 youngest tiles: the next tile has landed
    constexpr int WAIT_N = LPT * (NS - 2);
    constexpr int WAIT_IMM = 0x0F70 | (WAIT_N & 15) | ((WAIT_N >> 4) << 14);

    // Separate LDS objects (not one array indexed by stage): the compiler
    // then knows that the asynchronous global->LDS loads filling one buffer
    // cannot alias the fragment reads of another and does not serialise them.
    __shared__ __attribute__((aligned(2048))) unsigned char lds0[2 * TILE_BYTES];   // W tile, then X tile
    __shared__ __attribute__((aligned(2048))) unsigned char lds1[2 * TILE_BYTES];
    __shared__ __attribute__((aligned(2048))) unsigned char lds2[NS == 4 ? 2 * TILE_BYTES : 16];
    __shared__ __attribute__((aligned(2048))) unsigned char lds3[NS == 4 ? 2 * TILE_BYTES : 16];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);     // wave-uniform: keeps LDS bases scalar
    const int wn = wave >> 1, wm = wave & 1;
    const int l32 = lane & 31, g = lane >> 5;

    int tile_n, tile_m;
    tile_of_block(blockIdx.x, p.tiles_n * p.tiles_m, p.tiles_n, p.xn_parts, &tile_n, &tile_m);
    const int n0 = tile_n * BT, m0 = tile_m * BT;

    // ---- global -> LDS, asynchronous, no registers in between ----
    // One buffer_load ... lds instruction moves 64 lanes x 16 bytes = 16 tile rows
    // of one sub-block to 1 KiB of consecutive LDS (lane l lands at base + 16 l).
    // The wave's i-th load handles load number q = wave + 4 i of the tile:
    // sub-block q / SBDIV, 16-row group q % SBDIV.
    //   unpacked source: lane fetches row 16*group + l/4 and the chunk that belongs
    //     into LDS slot l%4, i.e. chunk (l%4) ^ swz(row); rows outside the matrix
    //     read as zero through the buffer descriptor's bounds check (which covers
    //     the lane offset only, so the row part lives there and just the K offset,
    //     always in range, goes into the scalar offset);
    //   packed source: the 1 KiB is contiguous in memory.
    const int KB = p.K * ES / 64;                    // 64-byte blocks per packed row
    const __amdgpu_buffer_rsrc_t wres = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<unsigned char*>(p.W), 0,
        p.w_packed ? (int)packed_bytes(p.N, p.K * ES) : (int)((size_t)p.N * p.K * ES), 0x00020000);
    const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<unsigned char*>(p.X), 0,
        p.x_packed ? (int)packed_bytes(p.M, p.K * ES) : (int)((((size_t)p.M - 1) * p.ldx + p.K) * ES), 0x00020000);
    const int w_rowb = p.K * ES, x_rowb = p.ldx * ES;
    const int dc = (lane & 3) ^ packed_swizzle(lane >> 2);     // row groups start at multiples of 16: only the lane matters
    const int w_base = p.w_packed ? ((n0 >> 8) * KB * 16384 + (n0 & 255) * 64 + wave * 1024 + lane * 16)
                                  : ((n0 + 16 * wave + (lane >> 2)) * w_rowb + (dc << 4));
    const int x_base = p.x_packed ? ((m0 >> 8) * KB * 16384 + (m0 & 255) * 64 + wave * 1024 + lane * 16)
                                  : ((m0 + 16 * wave + (lane >> 2)) * x_rowb + (dc << 4));
    const int w_gs = p.w_packed ? 1024 : 16 * w_rowb, w_ss = p.w_packed ? 16384 : 64;   // group / sub-block strides
    const int x_gs = p.x_packed ? 1024 : 16 * x_rowb, x_ss = p.x_packed ? 16384 : 64;
    const int w_ks = p.w_packed ? 32768 : 128, x_ks = p.x_packed ? 32768 : 128;         // K step strides

    typedef __attribute__((address_space(3))) void* lds_ptr_t;
    // K steps of this workgroup: all of them, or (split K) the blockIdx.y-th share
    const int steps = p.K / BK;
    const int kt0 = (int)((long)steps * blockIdx.y / p.splits);
    const int KT = (int)((long)steps * (blockIdx.y + 1) / p.splits);
    // A K step past the end (odd step counts run one phantom step) fetches from
    // beyond the descriptor's range and therefore fills the tile with zeros: bit 31 of
    // the lane offset puts it past any descriptor (launch_gemm keeps operands below 2 GiB).
#define CUBERT_ISSUE_TILE(BUF, kt)                                                                          \
    do {                                                                                                    \
        const int oob = (kt) < KT ? 0 : (int)0x80000000u;                                                   \
        _Pragma("unroll") for (int i = 0; i < GROUPS; ++i) {                                                \
            const int sb = (4 * i) / SBDIV, gq = (4 * i) % SBDIV;                                       \
            __builtin_amdgcn_raw_ptr_buffer_load_lds(                                                       \
                wres, (lds_ptr_t)((BUF) + sb * SUB + (gq + wave) * 1024), 16,                               \
                (w_base + gq * w_gs + sb * w_ss) | oob, (kt) * w_ks, 0, 0);                                 \
            __builtin_amdgcn_raw_ptr_buffer_load_lds(                                                       \
                xres, (lds_ptr_t)((BUF) + TILE_BYTES + sb * SUB + (gq + wave) * 1024), 16,                  \
                (x_base + gq * x_gs + sb * x_ss) | oob, (kt) * x_ks, 0, 0);                                 \
        }                                                                                                   \
    } while (0)

    // ---- fragment read addressing ----
    // Lane (row l32, group g) of 32x32 block i reads chunk 2*(kk&1) + g of row
    // base + 32 i + l32 in sub-block kk >> 1.  swz(row) only depends on l32 (the
    // quadrant base and 32 i do not reach the bits it uses), so the byte offset is
    //   (off0 ^ (kk & 1 ? kphase : 0)) + (kk >> 1) * SUB + i * 2048.
    const int woff0 = frag_base(wn * (BT / 2), p.w_units, l32, g), wkp = frag_kphase(p.w_units);
    const int xoff0 = TILE_BYTES + frag_base(wm * (BT / 2), p.x_units, l32, g), xkp = frag_kphase(p.x_units);

    f32x16_t acc[NB][NB];
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

    // With four stages the fragment reads are issued as inline asm on plain LDS byte addresses,
    // and waited for with an explicit lgkmcnt(0) that the fragments pass through ("+v"): a read
    // the compiler can see makes it wait for EVERY outstanding global->LDS load first, which
    // would undo the prefetch distance.  Which tile has landed is tracked by hand with the
    // vmcnt waits at the end of each step.  With two stages every load has landed at the end
    // of a step anyway and the compiler places the reads and their waits itself.
#define CUBERT_LOAD_FRAGS(BUF, kk, WF, XF)                                                                  \
    do {                                                                                                    \
        if constexpr (NS == 4) {                                                                            \
            const int cur = (int)(size_t)(__attribute__((address_space(3))) unsigned char*)(BUF);           \
            _Pragma("unroll") for (int i = 0; i < NB; ++i)                                                  \
                asm volatile("ds_read_b128 %0, %1" : "=v"(WF[i])                                            \
                             : "v"(cur + (wb ^ (((kk) & 1) ? wkp : 0)) + ((kk) >> 1) * SUB + i * 2048));         \
            _Pragma("unroll") for (int j = 0; j < NB; ++j)                                                  \
                asm volatile("ds_read_b128 %0, %1" : "=v"(XF[j])                                            \
                             : "v"(cur + (xb ^ (((kk) & 1) ? xkp : 0)) + ((kk) >> 1) * SUB + j * 2048));         \
        } else {                                                                                            \
            _Pragma("unroll") for (int i = 0; i < NB; ++i)                                                  \
                WF[i] = *reinterpret_cast<const u32x4_t*>((BUF) + (wb ^ (((kk) & 1) ? wkp : 0)) + ((kk) >> 1) * SUB + i * 2048); \
            _Pragma("unroll") for (int j = 0; j < NB; ++j)                                                  \
                XF[j] = *reinterpret_cast<const u32x4_t*>((BUF) + (xb ^ (((kk) & 1) ? xkp : 0)) + ((kk) >> 1) * SUB + j * 2048); \
        }                                                                                                   \
    } while (0)
#define CUBERT_FENCE_FRAGS(WF, XF)                                                                          \
    do {                                                                                                    \
        if constexpr (NS == 4) asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(WF[0]), "+v"(XF[0]));             \
    } while (0)

    // One K step on buffer CUR while the loads of the tile NS - 1 steps ahead fill NEXT
    // (the buffer the previous step computed on; its barrier has released it).
    // The empty asm keeps the compiler from hoisting (and then spilling) every
    // per-k-step address.
#define CUBERT_K_STEP(CUR, NEXT, kt)                                                                        \
    do {                                                                                                    \
        CUBERT_ISSUE_TILE(NEXT, (kt) + NS - 1);                                                             \
        int wb = woff0, xb = xoff0;                                                                         \
        asm volatile("" : "+v"(wb), "+v"(xb));                                                              \
        if constexpr (NS == 4) {                                                                            \
            /* One 32 x 32 block per wave: a k-slice is a single MFMA, too short to hide the next     */    \
            /* slice's fragment read behind it.  All eight reads of the step go out together and each */    \
            /* MFMA waits for its own pair only (LDS reads return in order).                          */    \
            u32x4_t wf[4][NB], xf[4][NB];                                                                   \
            _Pragma("unroll") for (int kk = 0; kk < 4; ++kk) CUBERT_LOAD_FRAGS(CUR, kk, wf[kk], xf[kk]);    \
            asm volatile("s_waitcnt lgkmcnt(6)" : "+v"(wf[0][0]), "+v"(xf[0][0]));                          \
            mfma_chunk<ELT>(wf[0][0], xf[0][0], acc[0][0]);                                                 \
            asm volatile("s_waitcnt lgkmcnt(4)" : "+v"(wf[1][0]), "+v"(xf[1][0]));                          \
            mfma_chunk<ELT>(wf[1][0], xf[1][0], acc[0][0]);                                                 \
            asm volatile("s_waitcnt lgkmcnt(2)" : "+v"(wf[2][0]), "+v"(xf[2][0]));                          \
            mfma_chunk<ELT>(wf[2][0], xf[2][0], acc[0][0]);                                                 \
            asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(wf[3][0]), "+v"(xf[3][0]));                          \
            mfma_chunk<ELT>(wf[3][0], xf[3][0], acc[0][0]);                                                 \
        } else {                                                                                            \
            u32x4_t wf[2][NB], xf[2][NB];                                                                   \
            CUBERT_LOAD_FRAGS(CUR, 0, wf[0], xf[0]);                                                        \
            CUBERT_FENCE_FRAGS(wf[0], xf[0]);                                                               \
            _Pragma("unroll") for (int kk = 0; kk < 4; ++kk) {                                              \
                if (kk < 3) CUBERT_LOAD_FRAGS(CUR, kk + 1, wf[(kk + 1) & 1], xf[(kk + 1) & 1]);             \
                _Pragma("unroll") for (int i = 0; i < NB; ++i)                                              \
                    _Pragma("unroll") for (int j = 0; j < NB; ++j)                                          \
                        mfma_chunk<ELT>(wf[kk & 1][i], xf[kk & 1][j], acc[i][j]);                           \
                if (kk < 3) CUBERT_FENCE_FRAGS(wf[(kk + 1) & 1], xf[(kk + 1) & 1]);                         \
            }                                                                                               \
        }                                                                                                   \
        __builtin_amdgcn_sched_barrier(0);  /* nothing moves across the end of the step */                  \
        __builtin_amdgcn_s_waitcnt(WAIT_IMM); /* my share of the next step's tile has landed */            \
        if constexpr (NS == 4) __builtin_amdgcn_s_barrier(); /* bare: a fenced one waits for all loads */  \
        else __syncthreads();                                                                               \
        __builtin_amdgcn_sched_barrier(0);                                                                  \
    } while (0)

    CUBERT_ISSUE_TILE(lds0, kt0);
    if constexpr (NS == 4) {
        CUBERT_ISSUE_TILE(lds1, kt0 + 1);
        CUBERT_ISSUE_TILE(lds2, kt0 + 2);
    }
    // The four-stage kernel runs launches of a few workgroups and a few K steps each, i.e. chains of round trips:
    // what the epilogue adds (bias, first residual rows) is requested now, behind the first tiles.
    constexpr bool SPLITK = (EPI == kEpiBias || EPI == kEpiBiasRes) && OUT == kF32;      // the only combinations launch_gemm splits
    constexpr bool PREFETCH = NS == 4 && BT == 64;
    f32x4_t bias[4 * NB];
    EpiPrefetch<EpiGeometry<OUT, EPI, NB, SPLITK, 4>::PB> pre;
    if constexpr (PREFETCH) {
        if constexpr (gemm_bias_at_readout<OUT, EPI>()) gemm_epilogue_prefetch<OUT, EPI, NB, SPLITK, 4>(p, n0 + wn * (BT / 2), m0 + wm * (BT / 2), l32, g, &pre);
        else gemm_load_bias<NB, SPLITK>(p, n0 + wn * (BT / 2), g, bias);
    }
    __builtin_amdgcn_s_waitcnt(WAIT_IMM);
    if constexpr (NS == 4) __builtin_amdgcn_s_barrier();
    else __syncthreads();
    if constexpr (NS == 4) {
        for (int kt = kt0; kt < KT; kt += 4) {
            CUBERT_K_STEP(lds0, lds3, kt);
            CUBERT_K_STEP(lds1, lds0, kt + 1);
            CUBERT_K_STEP(lds2, lds1, kt + 2);
            CUBERT_K_STEP(lds3, lds2, kt + 3);
        }
        // the zero tiles fetched past the end may still be landing in lds0, the epilogue's staging area
        __builtin_amdgcn_s_waitcnt(0x0F70);
        __syncthreads();
    } else {
        for (int kt = kt0; kt < KT; kt += 2) {
            CUBERT_K_STEP(lds0, lds1, kt);
            CUBERT_K_STEP(lds1, lds0, kt + 1);
        }
    }
#undef CUBERT_ISSUE_TILE
#undef CUBERT_LOAD_FRAGS
#undef CUBERT_FENCE_FRAGS
#undef CUBERT_K_STEP

    // (the larger tiles fetch their bias here rather than before the loop: no registers to spare there)
    if constexpr (!PREFETCH && !gemm_bias_at_readout<OUT, EPI>()) gemm_load_bias<NB, SPLITK>(p, n0 + wn * (BT / 2), g, bias);
    // every wave is past the last step's barrier: the tiles are dead, lds0 is free for staging
    gemm_epilogue<OUT, EPI, NB, NB, SPLITK, 4, true>(p, acc, bias, n0 + wn * (BT / 2), m0 + wm * (BT / 2), l32, g, lds0 + wave * (BT * 64),
                                                     PREFETCH && gemm_bias_at_readout<OUT, EPI>() ? &pre : nullptr);
}

template <int ELT, int OUT, int EPI, int BT, int NS = 2>
bool launch_one(const GemmDev& d, hipStream_t stream) {
    hipLaunchKernelGGL((gemm_kernel<ELT, OUT, EPI, BT, NS>), dim3(d.tiles_n * d.tiles_m, d.splits), dim3(256), 0, stream, d);
    CUBERT_HIP_OK(hipGetLastError());
    return true;
}

template <int ELT, int OUT, int EPI>
bool launch_tile(const GemmDev& d, int bt, hipStream_t stream) {
    switch (bt) {
        case 64:
            // few workgroups: nothing else on the CU hides the memory latency, so prefetch deeper
            if ((long)d.tiles_n * d.tiles_m * d.splits <= 512) return launch_one<ELT, OUT, EPI, 64, 4>(d, stream);
            return launch_one<ELT, OUT, EPI, 64>(d, stream);
        case 128: return launch_one<ELT, OUT, EPI, 128>(d, stream);
        case 256: return launch_one<ELT, OUT, EPI, 256>(d, stream);
    }
    set_error("gemm: tile must be 64, 128 or 256");
    return false;
}

template <int ELT, int OUT>
bool launch_epi(const GemmDev& d, int epi, int bt, hipStream_t stream) {
    switch (epi) {
        case kEpiBias: return launch_tile<ELT, OUT, kEpiBias>(d, bt, stream);
        case kEpiBiasGelu: return launch_tile<ELT, OUT, kEpiBiasGelu>(d, bt, stream);
        case kEpiBiasGeluUnits:
            if constexpr (OUT == kBF16) return launch_tile<ELT, OUT, kEpiBiasGeluUnits>(d, bt, stream);
            break;
        case kEpiBiasTanh: return launch_tile<ELT, OUT, kEpiBiasTanh>(d, bt, stream);
        case kEpiQKV: return launch_tile<ELT, OUT, kEpiQKV>(d, bt, stream);
        case kEpiQKVMap: return launch_tile<ELT, OUT, kEpiQKVMap>(d, bt, stream);
        case kEpiBiasRes:
            if constexpr (OUT == kF32) return launch_tile<ELT, OUT, kEpiBiasRes>(d, bt, stream);
            break;
    }
    set_error("gemm: unknown epilogue");
    return false;
}

}  // namespace

namespace {
// Workspace of the LayerNorm epilogue: flag words, two counters per band of rows (a fixed number of
// bands, so that launches with different M agree on where the counters are), then (sum, M2 about the slot mean)
// for every row and every 128-feature slot (at most 8).
constexpr size_t kLnMaxBands = 16384;
size_t ln_stats_offset() { return ((gemm_detail::kLnCntFirst + 2 * kLnMaxBands) * sizeof(int) + 255) / 256 * 256; }
}  // namespace

size_t gemm_ln_workspace_bytes(size_t M) { return ln_stats_offset() + ((M + 255) / 256 * 256) * 8 * sizeof(unsigned long long); }

namespace {
bool ln_shape_ok(int N, int K, int elt) { return elt == kBF16 && N > 0 && N % 256 == 0 && N <= 1024 && K % 32 == 0 && K >= 64; }
}  // namespace

bool gemm_ln_workspace_force_expiry(void* ln_ws) {
    if (!ln_ws) { set_error("gemm: null workspace"); return false; }
    const int limit = 1, stuck = -1000000;
    int* w = static_cast<int*>(ln_ws);
    CUBERT_HIP_OK(hipMemcpy(w + 1, &limit, sizeof(int), hipMemcpyHostToDevice));
    CUBERT_HIP_OK(hipMemcpy(w + gemm_detail::kLnCntFirst, &stuck, sizeof(int), hipMemcpyHostToDevice));
    return true;
}

// A launch gives every CU at most one workgroup if no XCD gets more workgroups than it has CUs: ln_tile_of_block hands out whole
// bands, band b and its N / 256 workgroups to XCD b % 8.  With N = 768, 81 to 85 bands are 243 to 255 workgroups, but 33 on up to
// five of the XCDs.
int gemm_ln_xcd_workgroups(int M, int N, int rows) {
    const int bands = (M + rows - 1) / rows;
    return (bands + 7) / 8 * (N / 256);
}

// Tile of a GEMM with the LayerNorm in its epilogue, 0 if the separate kernels are the better choice (below about 6000
// rows; N = 768 and 1024, K = N and 4 N).  The smallest tile that still makes one round of at most one workgroup per CU, since a
// launch lasts as long as its slowest CU; beyond that the 256 x 256 one.  Microseconds, cold weights, N = 1024, K = 1024 / 4096,
// with 128 / 192 / 256 tokens:  8192 rows 35.3 / 35.5 / 39.4 and 76.1 / 78.9 / 89.7;  8448 (264 tiles of 128 tokens) 43.4 / 36.6 /
// 39.9 and 101 / 81.2 / 90.3;  10947 48.5 / 41.2 / 43.8 and 112 / 89.6 / 96.6;  12288 51.3 / 44.0 / 45.7 and 116 / 96.4 / 99.9;
// 12416 (260 tiles of 192 tokens) 51.9 / 65.4 / 46.7 and 116 / 150 / 102.  N = 768, K = 768 / 3072:  10240 rows 30.0 / 32.5 / 37.2
// and 54.8 / 57.8 / 66.2;  10241 (81 bands of 128 tokens) 35.3 / 31.2 / 35.9 and 76.3 / 57.9 / 66.4;  12170 40.6 / 33.4 / 37.6 and
// 83.8 / 66.5 / 74.2;  15360 42.4 / 36.2 / 40.2 and 88.0 / 73.9 / 81.6;  15361 (81 bands of 192) 42.6 / 53.7 / 40.0 and 88.4 / 115 /
// 81.5.  The parts of a pass on two streams take the same tiles (18009 rows of BERT-large 12.76 ms against 12.80, 20926
// rows 15.17 against 15.27 with 256 tokens), except where those of the whole pass are one round (Model::ln_tile_of_parts).
int gemm_ln_pick_tile(int M, int N, int K, int elt) {
    if (M < 6144 || !ln_shape_ok(N, K, elt)) return 0;
    if (K % 128 != 0 || gemm_ln_xcd_workgroups(M, N, 128) <= kXcdCus) return kTile256x128;
    return gemm_ln_xcd_workgroups(M, N, 192) <= kXcdCus ? kTile256x192 : 256;
}

bool gemm_ln_supported(int M, int N, int K, int elt) { return gemm_ln_pick_tile(M, N, K, elt) != 0; }

int gemm_pick_tile(int M, int N, int K, int elt) {
    auto tiles = [&](int bt) { return (long)((M + bt - 1) / bt) * ((N + bt - 1) / bt); };
    auto rounds = [](long wgs, long slots) { return (double)((wgs + slots - 1) / slots); };
    if (elt != kBF16) {
        // float32 operands: a 128 tile keeps two workgroups on a CU, which the compiler-scheduled
        // loop needs more than the larger tile's operand reuse (measured 20 % faster than 256).
        return tiles(128) >= 512 ? 128 : 64;
    }
    // bf16: estimated time = rounds over the chip x time of one workgroup, with per-step costs
    // measured on MI355X (microseconds): the hand-scheduled 256 tile (one workgroup per CU)
    // 9 + 0.75 per 32 k; the hand-scheduled 256 x 128 tile (two per CU, which overlap instead of
    // running in rounds) 4.5 + 0.98 per 32 k (1.06 for K > 1536, where its shorter prefetch
    // distance shows); the 128 tile (two per CU) 5 + 1.2 per 64 k; the
    // 64 tile (four per CU) 4 + 0.9 per 64 k.
    const double c128 = rounds(tiles(128), 512) * (5.0 + 1.2 * K / 64.0);
    const double c64 = rounds(tiles(64), 1024) * (4.0 + 0.9 * K / 64.0);
    double best = c128;
    int bt = 128;
    if (c64 < best) { best = c64; bt = 64; }
    if (K % 128 == 0) {
        const double c256 = rounds(tiles(256), 256) * (9.0 + 0.75 * K / 32.0);
        if (c256 <= best) { best = c256; bt = 256; }
    }
    {
        const double wgs = (double)((M + 127) / 128) * ((N + 255) / 256);
        const double c384 = (wgs > 512.0 ? wgs / 512.0 : 1.0) * (4.5 + (K > 1536 ? 1.06 : 0.98) * K / 32.0);
        if (c384 < best) bt = kTile256x128;
    }
    return bt;
}

// Tile and split count for a problem (tile as in GemmParams::tile, never 0).  max_splits > 1: the caller can take the
// result as that many partial sums (float32 result, plain bias epilogue; see GemmParams::splits).
//
// Below kPlanSmallRows rows of bf16 operands the launch does not fill the chip for long and what counts is how the
// workgroups spread over the 256 CUs.  Estimated time (microseconds, constants measured on MI355X with launches of
// a few hundred to a few thousand rows of the four linears of BERT-large) = launch + result traffic + T * g, where T is the time of a
// workgroup that has its CU to itself (a constant plus a cost per half-step of 32 k), and g says how the launch
// stretches when a CU gets w > 1 workgroups on average: g = 1 + (w - 1 + q) * rho; rho is what one more workgroup on a CU
// costs relative to a lone one (1: nothing is gained from sharing a CU, the 128 x 128 tile saturates the LDS on its
// own) and q allows for the uneven hand-out of coarse tiles.  From kPlanSmallRows rows on gemm_pick_tile decides (its costs were
// measured inside whole forward passes at the power limit) and K is split only where 64 x 64 tiles would not give 512
// workgroups, which takes fewer output features than any BERT has.
constexpr int kPlanSmallRows = 6144;
constexpr int kShareFirst = 257;         // split operands: rows from which a tile whose four waves share K is chosen
constexpr int kShareRows = 8192;         // split operands: rows from which no tile whose waves share K is taken (a pass runs in parts there, in one k order)
// bf16: rows from and up to which mid_cost estimates, the latter for models from hidden 1024 on and for narrower ones; others: skinny_cost and the table in
// plan_small.  Passes of six layers, us, by those / by mid_cost:  from below, hidden 1024, 257 rows 295 / 284, 270 rows 299 / 284, 384 rows 333 / 314,
// hidden 640, 288 rows 233 / 235, 400 rows 278 / 263;  to above, hidden 1024, 1408 rows 566 / 542, 1536 rows 581 / 554, 1552 rows 603 / 608, 1800 rows
// 617 / 630;  hidden 768, 1536 rows 473 / 441, 2048 rows 506 / 478, 2400 rows 544 / 539, 2800 rows 603 / 603;  hidden 512, 2400 rows 439 / 435, 2800 rows
// 433 / 461.
constexpr int kMidFirst = 257, kMidLast = 1536, kMidLastNarrow = 2400;
// ... and the K from which, for float32 results (few features: a CU has one workgroup at most) and for others: below, a tile's estimate falls with the
// workgroups of a CU (the costs are fitted to K of 768 and more).  Passes of six layers, us, by mid_cost for every K / from these on: hidden 128, 800 to 1280
// rows 213 to 230 / 187 to 206, hidden 256, 1280 rows 263 / 241; hidden 384, 1280 rows, with 512 for both 277, with 384 for float32 results 269.
constexpr int kMidK = 512, kMidKF32 = 384;
// bf16: rows up to which a skinny tile is chosen (of narrow models: wider ones leave them before).  Hidden 64, us, with / without from 2048 rows on: 2560
// rows 212 / 215, 3200 223 / 224, 4000 235 / 234, 4800 251 / 246, 6080 269 / 263.
constexpr int kSkinnyLast = 4096;

namespace {
constexpr int kSkinnyTiles[] = {kTileSkinny11, kTileSkinny21, kTileSkinny12, kTileSkinny22};

// Estimated time (microseconds) of a launch of the skinny kernel.  q workgroups share the busiest CU.  Terms: what those fetch, at 148
// GB/s (64 bytes a clock), their MFMAs, the weights from memory at 6.1 TB/s, the result at 4 TB/s.  Least squares over launches of
// 17 to 400 rows of the four linears of BERT-base and BERT-large, each tile, 1 to 16 parts, halfway between weights from memory and
// weights in the L2 (mean error 6 %; the tile chosen by it is 1.2 % slower than the best in bf16, 0.2 % on split operands).
double skinny_cost(int M, int N, int K, bool split_operands, int tile, int sp, bool f32_result) {
    const int bn = skinny_features(tile), bm = skinny_tokens(tile), step = split_operands ? 16 : 32, es = split_operands ? 6 : 2;
    const long tiles = (long)((N + bn - 1) / bn) * ((M + bm - 1) / bm);
    const double q = (double)(((tiles + 7) / 8 * sp + kXcdCus - 1) / kXcdCus);
    const double k = (double)((K / step + 8 * sp - 1) / (8 * sp)) * 8 * step;      // of a workgroup, whole steps of its eight waves
    const double fetch = k * es * (bn + bm) / 148e3, weights = (double)N * K * es / 6.1e6, blocks = bn * bm / 1024.0;
    const double mfma = k / 16 * blocks * (split_operands ? 6 : 1) * 32 / 4 / 2400.0;
    const double out = (double)M * N * (f32_result ? 4.0 * sp : split_operands ? 6.0 : 2.0) / 4.0e6;
    return split_operands ? 2.47 + q * (1.25 * fetch + 0.61 * mfma + 2.48) - 2.48 + 0.33 * weights + 1.94 * out + 0.08 * (sp - 1)
                          : 1.67 + q * (1.08 * fetch + 0.73 * mfma) + 0.70 * weights + 0.135 * blocks + 4.03 * out + 0.02 * (sp - 1);
}

// The same for a few hundred to some two thousand rows (kMidFirst), the skinny tiles and the others on one scale.  w: workgroups per CU; a tile's time grows with w (1 at
// least), half-steps of 32 k and with how much of its last round is empty.  The skinny kernel as above, with what the average CU fetches beside
// the busiest one.  Least squares, then a search for the fewest microseconds lost by the choice, over 300 to 6000 rows of the four linears of
// BERT-base and BERT-large, every tile with 1 to 8 parts, weights from memory (40 matrices in turn), float32 results with the LayerNorm that
// adds the parts.  Up to 1280 rows the tile chosen is 0.6 % slower than the best on average (8 % at the worst), with the costs for fewer rows 8 % (39 %).
// Microseconds, LayerNorm included, their choice -> this one's:  FFN-out of BERT-base 1200 rows 22.0 -> 17.8, of BERT-large 800 rows 27.7 -> 22.1;
// attn-out of BERT-large 640 rows 12.5 -> 9.0, 1000 rows 12.3 -> 10.7.  Passes, pooled output on the host, 400 / 640 / 1024 / 1280 rows: BERT-base
// 526 -> 497, 586 -> 559, 696 -> 680, 730 -> 710; BERT-large 1350 -> 1309, 1640 -> 1587, 1858 -> 1818, 2286 -> 2199.
double mid_cost(int M, int N, int K, int tile, int bn, int bm, int sp, bool f32_result, bool gelu) {
    const double tiles = (double)((N + bn - 1) / bn) * ((M + bm - 1) / bm), w = tiles * sp / 256.0;
    const double out = (double)M * N * (f32_result ? 4.0 : 2.0) / 4.0e6, parts = (double)M * N * 4.0 * (sp - 1) / 4.0e6;
    if (is_skinny(tile)) {
        const double q = (double)((((long)tiles + 7) / 8 * sp + kXcdCus - 1) / kXcdCus), k = (double)((K / 32 + 8 * sp - 1) / (8 * sp)) * 256;
        const double fetch = k * 2 * (bn + bm) / 148e3, weights = (double)N * K * 2 / 6.1e6, blocks = bn * bm / 1024.0, mfma = k / 16 * blocks * 8 / 2400.0;
        return 0.732 + q * (0.829 * fetch + 0.431 * mfma + 0.459 * blocks - 0.352) + 0.843 * w * fetch + 1.15 * weights + 0.652 * out + 1.346 * parts;
    }
    struct Tile { int tile; double fixed, per_wg, per_hs, empty, empty_hs, deep_k, out, parts, gelu; };
    static const Tile costs[] = {
        {64, 4.271, -2.308, 0.158, 1.137, 0.03, -0.052, 1.559, 3.125, 0.094},
        {kTile128Hand, 8.238, -5.257, 0.327, 0.924, 0.018, -0.039, 1.256, 1.885, 0.165},
        {kTile256x128, 5.554, -0.844, 0.387, 0, 0.194, -0.053, 0.871, 0, 0.405},
        {kTile256x128Deep, 0.437, -1.31, 0.563, 7.845, 0.116, -0.204, 0.854, 0, 1.006},
        {256, 3.55, 1.415, 0.636, 10.54, 0.441, -0.105, 0.889, 0, 1.501},
    };
    const Tile* t = costs;
    while (t->tile != tile) ++t;
    const double g = w > 1.0 ? w : 1.0, empty = std::ceil(w) - g, hs = K / 32.0 / sp;
    // (a workgroup more on a CU takes time also at a K below those of the fit)
    const double one = t->per_wg + hs * (t->per_hs + (K > 2048 ? t->deep_k : 0.0)) + (gelu ? t->gelu : 0.0);
    return t->fixed + one + (g - 1.0) * std::max(one, 0.01 * hs) + empty * (t->empty + t->empty_hs * hs) + t->out * out + t->parts * parts;
}

// Best (tile, splits) with min_splits <= splits <= max_splits (powers of two times min_splits), all of one k order (kOrderAny:
// the operands and the epilogue suit the skinny kernel).
GemmPlan plan_small(int M, int N, int K, int min_splits, int max_splits, bool f32_result, bool gelu, int order) {
    // launch: before the first workgroup runs; fixed + per_hs * half-steps: a workgroup alone on its CU (deep_k: what a
    // half-step costs more when K > 2048 and the weights stream from memory); rho, q: see above; out: weight of the
    // result traffic (bytes / 4 TB/s).  Least-squares fit (5 % mean error) to launches of the four linears of BERT-large
    // at 400 .. 6400 rows that cycle through 40 weight matrices, so that weights come from memory as in a forward pass.
    struct Cand { int tile, bm, bn; double launch, fixed, per_hs, rho, q, out, deep_k; bool splits, k128; };
    static const Cand cands[] = {
        {64, 64, 64, 2.80, 0.20, 0.129, 0.77, 0.37, 0.01, 0.02, true, false},
        {kTile128Hand, 128, 128, 2.37, 2.81, 0.283, 0.61, 0.16, 0.28, 0.14, true, false},
        {kTile256x128, 128, 256, 8.00, 0.95, 0.260, 1.21, 0.45, 0.86, 0.46, false, false},
        {kTile256x128Deep, 128, 256, 6.25, 1.33, 0.263, 1.50, 0.62, 0.86, 0.43, false, true},
        {256, 256, 256, 8.00, 3.43, 0.448, 1.15, 0.85, 0.97, 0.11, false, true},
    };
    const bool mid = M >= kMidFirst && M <= (std::min(N, K) < 1024 ? kMidLastNarrow : kMidLast) && K >= (f32_result ? kMidKF32 : kMidK);
    GemmPlan best{order == kOrderSkinny ? (int)kTileSkinny12 : 64, min_splits};
    double best_cost = 1e30;
    for (const Cand& c : cands) {
        if (order == kOrderSkinny) break;
        if ((!c.splits && min_splits > 1) || (c.k128 && K % 128 != 0)) continue;
        for (int sp = min_splits; sp <= (c.splits ? max_splits : 1) && sp <= 16; sp *= 2) {
            if (sp > min_splits && K / sp < 128) break;             // at least four half-steps per share
            const double wgs = (double)((M + c.bm - 1) / c.bm) * ((N + c.bn - 1) / c.bn) * sp;
            const double w = wgs / 256.0;
            const double g = w <= 1.0 ? 1.0 : 1.0 + (w - 1.0 + c.q) * c.rho;
            const double T = c.fixed + c.per_hs * (K / 32.0 / sp) * (K > 2048 ? 1.0 + c.deep_k : 1.0) + (sp > 1 ? 0.6 : 0.0) +
                             (gelu ? 0.8 : 0.0);
            const double out_us = (double)M * N * (f32_result ? 4.0 : 2.0) * sp / 4.0e6;
            // the consumer of split results reads every part again
            const double cost = mid ? mid_cost(M, N, K, c.tile, c.bn, c.bm, sp, f32_result, gelu) : c.launch + c.out * out_us * (sp > 1 ? 1.5 : 1.0) + T * g;
            if (cost < best_cost) { best_cost = cost; best = GemmPlan{c.tile, sp}; }
        }
    }
    // The skinny tiles win up to a few hundred rows.  Microseconds, weights from memory / in the L2, best skinny tile against the best of
    // the others, attn-out and FFN-out with the LayerNorm that adds the parts.  BERT-base, QKV 17 rows 3.6 / 3.0 against 5.9 / 5.6,
    // 128 rows 4.4 / 3.7 against 6.3 / 5.9, 400 rows 5.7 / 4.9 against 6.1 / 5.8, 600 rows 8.9 / 8.1 against 8.5 / 7.8; FFN-out 17 rows
    // 6.9 / 6.0 against 8.3 / 7.5, 200 rows 9.7 / 8.9 against 10.5 / 9.9, 600 rows 13.1 / 13.2 against 13.9 / 14.2.  BERT-large, FFN-in
    // 128 rows 6.4 / 4.1 against 8.4 / 6.6, 200 rows 8.2 / 5.3 against 8.3 / 6.9, 400 rows 13.4 / 9.2 against 12.0 / 8.6; attn-out 128
    // rows 7.2 / 6.3 against 8.9 / 8.2, 600 rows 10.9 / 10.2 against 12.3 / 11.8.
    for (int tile : kSkinnyTiles) {
        if (order == kOrderShared || (order == kOrderAny && M > kSkinnyLast)) break;
        for (int sp = min_splits; sp <= max_splits && sp <= 16; sp *= 2) {
            if (4 * sp > K / 32 || (sp > min_splits && K / sp < 128)) break;
            const double cost = mid ? mid_cost(M, N, K, tile, skinny_features(tile), skinny_tokens(tile), sp, f32_result, gelu)
                                                    : skinny_cost(M, N, K, false, tile, sp, f32_result);
            if (cost < best_cost) { best_cost = cost; best = GemmPlan{tile, sp}; }
        }
    }
    return best;
}

// Estimated time (microseconds) of a launch on split operands, w workgroups per CU, on the scale of skinny_cost: of a tile whose four waves share K (one
// workgroup to a CU, so whole rounds, which last as long as their fetches and products; a round's GELU is not hidden), of 128 x 128 or of 256 x 128
// (two to a CU).  out: the result at 4 TB/s; parts: what the consumer reads beside the first part.  Least squares over 408 problems of 200 to 8100 rows of
// the four linears of hidden 256, 384, 512, 768 and 1024, 1 to 8 parts, weights from memory, float32 results with the LayerNorm that adds the parts,
// the competitive ones weighted most (mean error 6 %; what is chosen by it and skinny_cost is 1.4 % slower on average than the best).  A microsecond on
// all of them for the weights that a skinny tile finds in the L2s in a pass (l2_touch.h; with none, 1024 rows of BERT-large 985 us for six layers, with two
// 512 rows 658: 973 and 642 / 660 with one), and 3 % on tiles that share K beyond 4096 rows, where they are chosen too often otherwise.
double staged_or_share_cost(int M, int N, int K, int tile, int sp, double w, bool f32_result, bool gelu) {
    const double out = (double)M * N * (f32_result ? 4.0 : 6.0) / 4.0e6, parts = (double)M * N * 4.0 * (sp - 1) / 4.0e6, rounds = std::ceil(w);
    const double g = w > 1.0 ? w : 1.0, stretch = w > 1.0 ? rounds - g : 0.0;
    if (is_share(tile)) {
        const double blocks = share_features(tile) / 32, steps = (K / 16 + 4 * sp - 1) / (4 * sp);
        const double us = 3.3 + rounds * (steps * (0.391 + 0.299 * blocks) + (0.231 + (gelu ? 0.392 : 0.0)) * blocks) + 1.47 * out + 3.68 * parts;
        return M > 4096 ? 1.03 * us : us;
    }
    const double steps = K / 16.0 / sp;
    if (tile == kTile256x128) return 13.39 + g * (1.038 * steps - 8.02 + (gelu ? 3.2 : 0.0)) + 0.603 * stretch * steps + 0.632 * out;
    return 8.37 + g * (0.478 * steps - 2.6 + (gelu ? 1.22 : 0.0)) + 0.349 * stretch * steps + 0.836 * out + 2.71 * parts;
}

// float32 operands in the split layout.  Where tiles whose waves share K may be chosen (launches of a pass in one part), skinny_cost and
// staged_or_share_cost.  Best skinny tile / best share tile / 128 x 128 / 256 x 128, us, LayerNorm included:  BERT-large QKV 256 rows 16.2 / 17.5 / 33.2 / 74.1
// (share tiles are chosen from kShareFirst rows on), 400 rows 29.0 / 20.4 / 32.9 / 73.9, 1280 rows 59.9 / 45.5 / 43.5 / 74.4, 2048 rows 104.4 / 63.5 / 71.7 /
// 75.5, 5000 rows - / 152.4 / 141.5 / 139.3;  FFN-in of BERT-base 1408 rows 58.3 / 49.3 / 50.9 / 62.9, of BERT-large 1280 rows 79.8 / 62.4 / 71.4 / 78.0, 2048 rows
// 142.7 / 94.1 / 80.7 / 85.9;  FFN-out of BERT-base 1024 rows 42.2 / 33.0 / 39.1 / -, 1280 rows 44.0 / 38.2 / 44.3 / -.  (With 256 x 128 on the scale below, which
// knows no GELU and no result, FFN-in took it from 1280 rows on;
// passes of six layers, us, before / now: BERT-large 1280 rows 1251 / 1191, 1408 rows 1386 / 1332, BERT-base 1408 rows 980 / 956, 2048 rows 1197 / 1142.)
// Otherwise the time of a workgroup alone on its CU, stretched by w = workgroups / 256 (cold weights, up to 19600 rows):
//   (fixed + per_step * 16-k steps) * (w > 1 ? w + 0.5 : 1): a second workgroup on a CU costs nearly what the first did, and the hand-out is uneven by
//   half a workgroup; 256 x 128 wins from about 900 tiles on.  The constants of 128 x 128 are those of its loop before it read fragments a step
//   ahead (gemm_split.hip), which takes less from launches of few workgroups.
GemmPlan plan_split_operands(int M, int N, int K, int min_splits, int max_splits, bool f32_result, bool gelu, int order) {
    struct Cand { int tile, bm, bn; double fixed, per_step; int order; };
    static const Cand cands[] = {
        {128, 128, 128, 6.0, 0.455, kOrderShared},
        {kTile256x128, 128, 256, 8.0, 0.98, kOrderShared},
        {kTileSkinny11, 0, 0, 0.0, 0.0, kOrderSkinny},
        {kTileSkinny21, 0, 0, 0.0, 0.0, kOrderSkinny},
        {kTileSkinny12, 0, 0, 0.0, 0.0, kOrderSkinny},
        {kTileSkinny22, 0, 0, 0.0, 0.0, kOrderSkinny},
        {kTileShare1, 128, 32, 0.0, 0.0, kOrderShare4},
        {kTileShare2, 128, 64, 0.0, 0.0, kOrderShare4},
        {kTileShare3, 128, 96, 0.0, 0.0, kOrderShare4},
    };
    GemmPlan best{order == kOrderSkinny ? (int)kTileSkinny12 : order == kOrderShare4 ? (int)kTileShare3 : 128, min_splits};
    double best_cost = 1e30;
    for (const Cand& c : cands) {
        if (order != kOrderAny && order != c.order) continue;
        const bool skinny = c.order == kOrderSkinny;
        if (skinny && (N % 8 != 0 || split_bytes(M, K) >= (1ull << 31) || split_bytes(N, K) >= (1ull << 31))) continue;
        if (c.order == kOrderShare4 && ((order == kOrderAny && M < kShareFirst) || (N + c.bn - 1) / c.bn > 65535)) continue;      // (65535: what its kernel numbers)
        for (int sp = min_splits; sp <= max_splits && sp <= 16; sp *= 2) {
            if (sp > min_splits && K / sp < 128) break;
            if (c.order != kOrderShared && 4 * sp > K / 16) break;
            if (c.tile == kTile256x128 && sp > 1 && order != kOrderShared) break;          // staged_or_share_cost knows it whole only
            double cost;
            if (skinny) {
                cost = skinny_cost(M, N, K, true, c.tile, sp, f32_result);
            } else {
                const double w = (double)((M + c.bm - 1) / c.bm) * ((N + c.bn - 1) / c.bn) * sp / 256.0, g = w > 1.0 ? w + 0.5 : 1.0;
                if (order != kOrderShared) {
                    cost = staged_or_share_cost(M, N, K, c.tile, sp, w, f32_result, gelu);
                } else {
                    cost = (c.fixed + c.per_step * (K / 16.0 / sp)) * (w > 4.0 && c.tile == kTile256x128 ? w : g);
                    // every part of a split result is written and read again by the consumer
                    if (sp > 1) cost += 0.6 + (double)M * N * 4.0 * sp / 4.0e6;
                }
            }
            if (cost < best_cost) { best_cost = cost; best = GemmPlan{c.tile, sp}; }
        }
    }
    return best;
}

// Launches a GEMM on split operands.
bool launch_split_operands(const GemmParams& p, hipStream_t stream) {
    if (p.M <= 0 || p.N <= 0 || p.K <= 0 || p.K % 16 != 0 || p.N % 4 != 0) { set_error("gemm: split operands need K to be a multiple of 16 and N of 4"); return false; }
    if (!p.X || !p.W || !p.bias || ((reinterpret_cast<uintptr_t>(p.X) | reinterpret_cast<uintptr_t>(p.W) | reinterpret_cast<uintptr_t>(p.bias)) & 15)) {
        set_error("gemm: null or misaligned operand");
        return false;
    }
    if ((size_t)p.K * 6 * 256 >= (1ull << 31)) { set_error("gemm: K too large"); return false; }
    if (p.ln_gamma || p.compiler_scheduled || (p.tile != 0 && p.tile != 128 && p.tile != kTile256x128 && !is_skinny(p.tile) && !is_share(p.tile))) {
        set_error("gemm: split operands take the 128, the 256x128 or a tile whose waves share K and no LayerNorm epilogue");
        return false;
    }
    GemmDev d{};
    d.X = static_cast<const unsigned char*>(p.X);
    d.W = static_cast<const unsigned char*>(p.W);
    d.bias = p.bias;
    d.Y = static_cast<unsigned char*>(p.Y);
    d.M = p.M; d.N = p.N; d.K = p.K; d.ldx = p.K;
    d.splits = p.splits > 0 ? p.splits : 1;
    int epi = p.epilogue;
    if (epi == kEpiQKV) {
        if (!p.q || !p.k || !p.vt || p.S <= 0 || p.heads <= 0 || p.N != 3 * p.heads * 64 || (!p.rowmap && p.M % p.S != 0) ||
            p.Sp < p.S || p.Sp % 32 != 0 || p.residual || d.splits > 1) {
            set_error("gemm: bad QKV epilogue arguments");
            return false;
        }
        d.q = static_cast<unsigned char*>(p.q);
        d.k = static_cast<unsigned char*>(p.k);
        d.vt = static_cast<unsigned char*>(p.vt);
        d.S = p.S; d.Sp = p.Sp; d.heads = p.heads; d.hidden = p.heads * 64;
        d.rowmap = p.rowmap;
        if (p.rowmap) epi = kEpiQKVMap;
    } else {
        if (!p.Y || (reinterpret_cast<uintptr_t>(p.Y) & 15)) { set_error("gemm: bad Y"); return false; }
        if (epi == kEpiBiasGelu ? (p.out_elt != kF32Split || p.N % 32 != 0 || p.residual || d.splits > 1) : (epi != kEpiBias || p.out_elt != kF32)) {
            set_error("gemm: split operands give float32 results (bias, residual) or split ones (GELU, N a multiple of 32)");
            return false;
        }
        if (p.residual) {
            if (reinterpret_cast<uintptr_t>(p.residual) & 15) { set_error("gemm: misaligned residual"); return false; }
            epi = kEpiBiasRes;
            d.R = p.residual;
        }
    }
    const int tile = p.tile ? p.tile : plan_split_operands(p.M, p.N, p.K, d.splits, d.splits, p.out_elt == kF32 && epi != kEpiQKV && epi != kEpiQKVMap, epi == kEpiBiasGelu, p.k_order).tile;
    if (is_skinny(tile)) {
        if (split_bytes(p.M, p.K) >= (1ull << 31) || split_bytes(p.N, p.K) >= (1ull << 31)) {
            set_error("gemm: operand exceeds the 2 GiB addressable through one buffer descriptor");
            return false;
        }
        d.xn_parts = p.xcd_partition > 0 ? p.xcd_partition : 0;
        return launch_gemm_skinny(d, kF32Split, tile, epi, stream);
    }
    const int bn = is_share(tile) ? share_features(tile) : tile == kTile256x128 ? 256 : 128;
    d.tiles_n = (p.N + bn - 1) / bn;
    d.tiles_m = (p.M + 127) / 128;
    d.xn_parts = gemm_pick_partition((double)p.M * p.K * 6, (double)p.N * p.K * 6, d.tiles_n, d.tiles_m, 8);
    if (p.xcd_partition >= 0) d.xn_parts = p.xcd_partition;
    return is_share(tile) ? launch_gemm_split_share(d, tile, epi, stream) : launch_gemm_split(d, tile, epi, stream);
}
}  // namespace

GemmPlan gemm_plan(int M, int N, int K, int elt, int max_splits, bool f32_result, bool gelu, bool any_order) {
    const int order = any_order && N % 8 == 0 ? kOrderAny : kOrderShared;
    if (elt == kF32Split) return plan_split_operands(M, N, K, 1, max_splits > 1 ? max_splits : 1, f32_result, gelu, M < kShareRows ? order : (int)kOrderShared);
    GemmPlan best{gemm_pick_tile(M, N, K, elt), 1};
    if (elt != kBF16 || M >= kPlanSmallRows || K % 64 != 0) {
        if (max_splits > 1) {
            // many rows and few features, or a K that plan_small's tiles do not take: at most 512 workgroups of 64 x 64 tiles
            const long tiles = (long)((M + 63) / 64) * ((N + 63) / 64);
            int sp = 1;
            while (sp * 2 <= max_splits && tiles * sp < 512 && K / (sp * 2) >= 256) sp *= 2;
            best.splits = sp;
            if (sp > 1 && best.tile == 256) best.tile = 128;      // the 256 x 256 kernel does not split
        }
        return best;
    }
    return plan_small(M, N, K, 1, max_splits > 1 ? max_splits : 1, f32_result, gelu, order);
}

bool launch_gemm(const GemmParams& p, hipStream_t stream) {
    if (p.xcd_partition != -1 && p.xcd_partition != 0 && p.xcd_partition != 2 && p.xcd_partition != 4) { set_error("gemm: the XCD partition is 0, 2 or 4"); return false; }
    if (p.elt == kF32Split) return launch_split_operands(p, stream);
    const int es = (p.elt == kBF16) ? 2 : 4;
    const int bk = 128 / es;
    if (p.elt != kBF16 && p.elt != kF32) { set_error("gemm: bad operand type"); return false; }
    if (p.M <= 0 || p.N <= 0 || p.K <= 0) { set_error("gemm: empty problem"); return false; }
    if (p.K % bk != 0) { set_error("gemm: K must be a multiple of " + std::to_string(bk)); return false; }
    if (p.N % 4 != 0) { set_error("gemm: N must be a multiple of 4"); return false; }
    if (p.out_elt == kBF16 && p.N % 8 != 0) { set_error("gemm: N must be a multiple of 8 for bf16 results"); return false; }
    if (!p.x_packed && (p.ldx < p.K || (p.ldx * es) % 16 != 0)) { set_error("gemm: bad ldx"); return false; }
    if (p.x_packed && p.ldx != p.K) { set_error("gemm: a packed X has no row stride"); return false; }
    if (!p.X || !p.W || !p.bias) { set_error("gemm: null operand"); return false; }
    if (((size_t)p.M + 256) * (p.x_packed ? p.K : p.ldx) * es >= (1ull << 31) ||
        ((size_t)p.N + 256) * p.K * es >= (1ull << 31)) {
        set_error("gemm: operand exceeds the 2 GiB addressable through one buffer descriptor");
        return false;
    }
    if ((reinterpret_cast<uintptr_t>(p.X) | reinterpret_cast<uintptr_t>(p.W) |
         reinterpret_cast<uintptr_t>(p.bias)) & 15) {
        set_error("gemm: operands must be 16-byte aligned");
        return false;
    }
    GemmDev d{};
    d.X = static_cast<const unsigned char*>(p.X);
    d.W = static_cast<const unsigned char*>(p.W);
    d.bias = p.bias;
    d.Y = static_cast<unsigned char*>(p.Y);
    d.M = p.M; d.N = p.N; d.K = p.K; d.ldx = p.ldx;
    d.x_packed = p.x_packed; d.w_packed = p.w_packed; d.y_packed = p.y_packed;
    d.x_units = p.x_units; d.w_units = p.w_units; d.y_units = p.y_units;
    if ((p.x_units && !p.x_packed) || (p.w_units && !p.w_packed) || (p.y_units && !p.y_packed) || ((p.x_units || p.w_units) && p.elt != kBF16)) {
        set_error("gemm: the units layout is a packed layout of bf16 operands");
        return false;
    }
    int out = p.out_elt;
    int epi = (p.epilogue == kEpiQKV && p.rowmap) ? (int)kEpiQKVMap : p.epilogue;
    if (p.epilogue == kEpiQKVMap || p.epilogue == kEpiBiasRes || p.epilogue == kEpiBiasResLN || p.epilogue == kEpiBiasGeluUnits) { set_error("gemm: unknown epilogue"); return false; }
    if (p.residual) {
        if (p.epilogue != kEpiBias || out != kF32 || p.y_packed || p.N % 4 != 0 ||
            (reinterpret_cast<uintptr_t>(p.residual) & 15)) {
            set_error("gemm: a residual needs the plain bias epilogue, a float32 row-major result, N a multiple of 4 and 16-byte alignment");
            return false;
        }
        epi = kEpiBiasRes;
        d.R = p.residual;
    }
    if (p.ln_gamma) {
        if (!p.residual || !p.ln_beta || !p.ln_ws || p.splits > 1 || !ln_shape_ok(p.N, p.K, p.elt) ||
            ((size_t)p.M + 256) * p.N * 4 >= (1ull << 31) || (size_t)(p.M + 127) / 128 > kLnMaxBands ||
            (p.tile ? (p.tile != 256 && p.tile != kTile256x192 && p.tile != kTile256x128) || (p.tile != kTile256x128 && p.K % 128 != 0)
                    : !gemm_ln_supported(p.M, p.N, p.K, p.elt)) ||
            ((reinterpret_cast<uintptr_t>(p.ln_gamma) | reinterpret_cast<uintptr_t>(p.ln_beta) |
              reinterpret_cast<uintptr_t>(p.ln_xb) | reinterpret_cast<uintptr_t>(p.ln_ws)) & 15)) {
            set_error("gemm: the LayerNorm epilogue needs a residual, bf16 operands, N a multiple of 256 up to 1024, the "
                      "256, 256x192 or 256x128 tile, no split K, a workspace and 16-byte aligned gamma / beta / copy");
            return false;
        }
        epi = kEpiBiasResLN;
        d.ln_gamma = p.ln_gamma;
        d.ln_beta = p.ln_beta;
        d.ln_xb = static_cast<unsigned char*>(p.ln_xb);
        d.ln_xb_packed = p.ln_xb_packed ? 1 : 0;
        d.ln_bands = (int)kLnMaxBands;
        d.ln_cnt = static_cast<int*>(p.ln_ws);
        d.ln_stats = reinterpret_cast<unsigned long long*>(static_cast<unsigned char*>(p.ln_ws) + ln_stats_offset());
    }
    if (p.epilogue == kEpiQKV) {
        if (!p.q || !p.k || !p.vt || p.S <= 0 || p.heads <= 0 || p.N != 3 * p.heads * 64 ||
            (!p.rowmap && p.M % p.S != 0) || p.Sp < p.S || p.Sp % 4 != 0) {
            set_error("gemm: bad QKV epilogue arguments");
            return false;
        }
        d.q = static_cast<unsigned char*>(p.q);
        d.k = static_cast<unsigned char*>(p.k);
        d.vt = static_cast<unsigned char*>(p.vt);
        d.v_rowmajor = p.v_rowmajor ? 1 : 0;
        d.S = p.S; d.Sp = p.Sp; d.heads = p.heads; d.hidden = p.heads * 64;
        d.rowmap = p.rowmap;
        d.y_packed = d.y_units = 0;
        out = p.elt;
    } else {
        if (!p.Y || (reinterpret_cast<uintptr_t>(p.Y) & 15)) { set_error("gemm: bad Y"); return false; }
        if (out != kBF16 && out != kF32) { set_error("gemm: bad output type"); return false; }
        if (p.y_units && epi == kEpiBiasGelu) epi = kEpiBiasGeluUnits;
        if (p.y_packed && (out != kBF16 || p.N % 32 != 0 || (p.y_units && epi != kEpiBiasGeluUnits))) {
            set_error("gemm: a packed Y must be bf16 with N a multiple of 32");
            return false;
        }
    }
    d.splits = p.splits > 0 ? p.splits : 1;
    if (d.splits > 1) {
        if ((epi != kEpiBias && epi != kEpiBiasRes) || out != kF32 || p.y_packed || d.splits > p.K / bk) {
            set_error("gemm: split K needs the plain bias epilogue, a float32 result and at least one K step per split");
            return false;
        }
    }
    // what the skinny kernel reads and writes, whoever asks for its tile (which those who do not want V row-major may not)
    const bool skinny_fits = p.elt == kBF16 && p.x_units && p.w_units && p.N % 8 == 0 &&
                             (p.epilogue == kEpiQKV ? p.v_rowmajor || !p.tile : epi == kEpiBiasGeluUnits || ((epi == kEpiBias || epi == kEpiBiasRes) && out == kF32));
    int bt = p.tile;
    if (!bt) {
        // the caller has settled on the split count; the tile follows
        if (p.k_order == kOrderSkinny || (p.elt == kBF16 && p.M < kPlanSmallRows && p.K % 64 == 0)) {
            const int order = p.k_order == kOrderAny && (!skinny_fits || p.compiler_scheduled) ? (int)kOrderShared : p.k_order;
            bt = plan_small(p.M, p.N, p.K, d.splits, d.splits, out == kF32, p.epilogue == kEpiBiasGelu, order).tile;
        }
        else
            bt = gemm_pick_tile(p.M, p.N, p.K, p.elt);
    }
    if (epi == kEpiBiasResLN && !p.tile) bt = gemm_ln_pick_tile(p.M, p.N, p.K, p.elt);
    if (d.splits > 1 && (bt == 256 || bt == kTile256x128 || bt == kTile256x128Deep) && !p.tile) bt = 128;      // those kernels do not split
    if (epi == kEpiBiasResLN && p.compiler_scheduled) { set_error("gemm: the LayerNorm epilogue has no compiler-scheduled kernel"); return false; }
    if (bt == kTile256x192) {
        if (epi != kEpiBiasResLN) { set_error("gemm: the 256x192 tile is there for the LayerNorm epilogue only"); return false; }
        d.tiles_n = p.N / 256;
        d.tiles_m = (p.M + 191) / 192;
        return launch_gemm_bf16_t256x192_ln(d, stream);
    }
    if (bt == kTile256x128 || bt == kTile256x128Deep) {
        if (p.elt != kBF16 || d.splits != 1) { set_error("gemm: the 256x128 tile is bf16 only and does not split K"); return false; }
        d.tiles_n = (p.N + 255) / 256;
        d.tiles_m = (p.M + 127) / 128;
        d.xn_parts = gemm_pick_partition((double)p.M * p.K * es, (double)p.N * p.K * es, d.tiles_n, d.tiles_m, 8);
        if (p.xcd_partition >= 0) d.xn_parts = p.xcd_partition;
        if (bt == kTile256x128Deep) {
            if (epi == kEpiBiasResLN) { set_error("gemm: the one-per-CU 256x128 tile has no LayerNorm epilogue"); return false; }
            return launch_gemm_bf16_t256x128_deep(d, out, epi, stream);
        }
        return launch_gemm_bf16_t256x128(d, out, epi, stream);
    }
    if (is_skinny(bt)) {
        if (!skinny_fits) {
            set_error("gemm: the skinny tiles need bf16 operands in the units layout and a GELU result in it, row-major QKV or float32 result");
            return false;
        }
        d.xn_parts = p.xcd_partition > 0 ? p.xcd_partition : 0;
        return launch_gemm_skinny(d, kBF16, bt, epi == kEpiBiasGeluUnits ? (int)kEpiBiasGelu : epi, stream);
    }
    if (bt == kTile128Hand) {
        if (p.elt != kBF16) { set_error("gemm: the hand-scheduled 128 tile is bf16 only"); return false; }
        d.tiles_n = (p.N + 127) / 128;
        d.tiles_m = (p.M + 127) / 128;
        d.xn_parts = gemm_pick_partition((double)p.M * p.K * es, (double)p.N * p.K * es, d.tiles_n, d.tiles_m, 8);
        if (p.xcd_partition >= 0) d.xn_parts = p.xcd_partition;
        return launch_gemm_bf16_t128(d, out, epi, stream);
    }
    d.tiles_n = (p.N + bt - 1) / bt;
    d.tiles_m = (p.M + bt - 1) / bt;
    d.xn_parts = gemm_pick_partition((double)p.M * p.K * es, (double)p.N * p.K * es, d.tiles_n, d.tiles_m, 4);
    if (p.xcd_partition >= 0) d.xn_parts = p.xcd_partition;
    if (p.elt == kBF16) {
        // 256 tile with a multiple of four half-steps: the hand-scheduled kernel
        if (bt == 256 && p.K % 128 == 0 && !p.compiler_scheduled && d.splits == 1)
            return launch_gemm_bf16_t256(d, out, epi, stream);
        return out == kBF16 ? launch_epi<kBF16, kBF16>(d, epi, bt, stream)
                            : launch_epi<kBF16, kF32>(d, epi, bt, stream);
    }
    if (out != kF32) { set_error("gemm: f32 operands require f32 output"); return false; }
    return launch_epi<kF32, kF32>(d, epi, bt, stream);
}

}  // namespace cubert
