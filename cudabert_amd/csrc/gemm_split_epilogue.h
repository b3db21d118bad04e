// Epilogue of the kernels on split operands (gemm_split.hip, gemm_split_share.hip).
#pragma once
#include "gemm_common.h"

namespace cubert {
namespace gemm_detail {

// Epilogues whose result is an operand in MFMA register layout: bias + GELU in the split layout (the next GEMM's operand), and
// Q, K, V as the attention kernel reads them.  split_unit_rows turns accumulator layout into 16 bytes per lane and plane;
// they leave in 1 KiB units (Q, K, V: two runs of up to 512 bytes) without a trip through the LDS.
template <int EPI, int NBI, int NBJ>
__device__ __forceinline__ void split_epilogue(const GemmDev& p, f32x16_t (&acc)[NBI][NBJ], const f32x4_t (&bias)[4 * NBI],
                                               int n_base, int m_base, int l32, int g) {
    const int row_blocks = (p.M + 31) / 32, nblk = p.Sp >> 5;
#pragma unroll
    for (int j = 0; j < NBJ; ++j) {
        const int rb = (m_base >> 5) + j;
        if (rb >= row_blocks) continue;                    // wave-uniform
        const int m = m_base + 32 * j + l32;
        int bidx = 0, sidx = 0;
        if constexpr (EPI != kEpiBiasGelu) {
            const int mc = m < p.M ? m : p.M - 1;
            const int tok = EPI == kEpiQKVMap ? p.rowmap[mc] : mc;
            bidx = tok / p.S;
            sidx = tok - bidx * p.S;
        }
#pragma unroll
        for (int i = 0; i < NBI; ++i) {
            if (n_base + 32 * i >= p.N) continue;          // N % 32 == 0
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int n = n_base + 32 * i + 16 * u;
                float x[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    x[e] = acc[i][j][8 * u + e] + bias[4 * i + 2 * u + e / 4][e % 4];
                    if constexpr (EPI == kEpiBiasGelu) x[e] = gelu_erf(x[e]);
                }
                u32x4_t pl[3];
                split_unit_rows(x, pl);
                unsigned char* dst;
                if constexpr (EPI == kEpiBiasGelu) {
                    dst = p.Y + ((size_t)rb * (p.N / 16) + n / 16) * 3072 + (l32 + 32 * g) * 16;
                } else {
                    const int which = n >= 2 * p.hidden ? 2 : n >= p.hidden ? 1 : 0;
                    const int hn = n - which * p.hidden, kk = (hn & 63) >> 4, pos = sidx & 31;
                    const size_t unit = ((((size_t)bidx * p.heads + (hn >> 6)) * nblk + (sidx >> 5)) * 4 + kk) * 3;
                    dst = (which == 2 ? p.vt : which ? p.k : p.q) + unit * 1024 + g * 512 + (which == 2 ? attn_v_slot(pos, g, kk) : pos) * 16;
                    if (m >= p.M) continue;
                }
#pragma unroll
                for (int q = 0; q < 3; ++q) *reinterpret_cast<u32x4_t*>(dst + q * 1024) = pl[q];
            }
        }
    }
}

}  // namespace gemm_detail
}  // namespace cubert
