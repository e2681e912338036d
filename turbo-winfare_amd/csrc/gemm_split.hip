// Batched (B > 2) affine-int4 LM head for tables with few 64-row tiles, on the matrix cores.
//
// The head of gemm_mfma.hip gives a wave a whole tile: with a few hundred tiles most of the 256
// CUs stay idle and each wave walks all groups one after another, bound by the latency of its own
// loads. Here the KS waves of a workgroup share one tile and 32 batch columns and split the
// groups, wave w taking [w G / KS, (w + 1) G / KS). Nothing is shared between the waves while they
// stream (no barrier, no LDS ring): each reads its groups' weights and its activation fragments
// straight into registers, PF groups ahead, the activations from a fragment-ordered copy (one
// contiguous 1 KiB per fragment, written by the step prep). The partial tiles then go through LDS,
// are added in wave order, and the epilogue takes one column per wave, lane = row.
#include <hip/hip_ext.h>

#include <stdexcept>

#include "dt_mfma.h"

namespace tdt {

// Floats of one column of a partial tile in LDS: 64 rows and 4 of padding, so that the
// accumulators' 16-byte stores (16 lanes = 16 columns) fall in distinct banks.
constexpr uint32_t kPartCol = 68;

// One column's 64 raw sums, lane = row: row scale, softcap, modifiers, ban, then the logit and the
// block summary. mw: the column's modifier words, as staged by the kernel.
__device__ inline void split_column(float l, uint32_t b, uint32_t tile, uint32_t lane, const uint32_t (&mw)[10],
                                    const EpiArgs& ep) {
#pragma clang fp contract(off)
    const uint32_t id = tile * kTileRows + lane, hl = lane >> 5, l32 = lane & 31u;
    const bool valid = id < ep.V;
    if (ep.xscale) l = l * ep.xscale[b];  // undoes the row's fp16 scaling (a power of two)
    if (ep.cap > 0.0f) l = ep.cap * tanhf(l / ep.cap);
    if (ep.meta) {
        const uint32_t has_mods = mw[0];
        if (has_mods && valid) {
            DevRow row{};
            row.repetition_penalty = __uint_as_float(mw[1]);
            row.presence_penalty = __uint_as_float(mw[2]);
            row.frequency_penalty = __uint_as_float(mw[3]);
            ModEntry m{id, 0u, 0.0f, 0u};
            if ((has_mods & 1u) && ep.hcount) {
                const uint32_t hw = mw[4u + hl];
                if (l32 == 0u && hw != 0u) ep.hbits[(size_t)b * ep.hbw + (id >> 5)] = 0u;
                if ((hw >> l32) & 1u) {
                    uint32_t* cp = ep.hcount + (size_t)b * ep.V + id;
                    m.count = *cp;
                    if (m.count) *cp = 0u;  // stored after the load it depends on
                }
            }
            if ((has_mods & 2u) && ep.block_start) {
                const ModEntry* me = ep.mods + (size_t)b * ep.mod_cap;
                for (uint32_t k = mw[8]; k < mw[9]; ++k) {
                    const ModEntry t = me[k];
                    if (t.id == id) { m.bias = t.bias; m.has_bias = 1u; }
                }
            }
            if (m.count || m.has_bias) l = apply_entry(l, m, row, ep.rep_limit);
        }
        if (ep.ban && ((mw[6u + hl] >> l32) & 1u)) l = -INFINITY;
    }
    finish_value(l, b, tile, lane, ep);
}

template <int KS, bool DENORM>
__global__ __launch_bounds__(64 * KS, 4) void k_head_mfma_split(
    const uint4* __restrict__ Wt, const uint32_t* __restrict__ SB16t, const uint16_t* __restrict__ xf, uint32_t B,
    uint32_t NC, uint32_t G, uint32_t ncb, EpiArgs ep) {
    constexpr int PF = 2;
    __shared__ __attribute__((aligned(16))) float part[KS][32 * kPartCol];
    __shared__ uint32_t meta[32][10];
    const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t hl = lane >> 5, l32 = lane & 31u;
    // the column blocks of one tile on one XCD, back to back (gemm_mfma.hip)
    const uint32_t wg = blockIdx.x, xcd = wg & 7u, slot = wg >> 3;
    const uint32_t tile = (slot / ncb) * 8u + xcd, cb = slot % ncb;
    if (tile >= ep.ntile) return;  // padding: ntile rounded up to 8
    const uint32_t cbase = 32u * cb;
    const uint32_t g0 = wave * G / KS, g1 = (wave + 1u) * G / KS;  // empty when KS > G

    const __amdgpu_buffer_rsrc_t wrs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint4*>(Wt), 0, ep.ntile * NC * kTileRows * 16u, kBufDword3);
    const __amdgpu_buffer_rsrc_t srs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(SB16t), 0, ep.ntile * G * kTileRows * 4u, kBufDword3);
    const uint32_t xbytes = G * ncb * 4096u;
    const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(xf), 0, xbytes, kBufDword3);
    const uint32_t woff = ((tile * NC + hl) * kTileRows + l32) * 16u;
    const uint32_t soff = (tile * G * kTileRows + l32) * 4u;
    // columns past the batch read past the buffer's end: zeros, and no traffic
    const uint32_t xoff = (cbase + l32 < B) ? cb * 4096u + lane * 16u : xbytes;
    const uint32_t magic = DENORM ? 0u : magic_vgpr();

    // the modifier words of this tile's columns (one thread each), stored to LDS after the loop
    uint32_t mt[10];
#pragma unroll
    for (int k = 0; k < 10; ++k) mt[k] = 0u;
    if (ep.meta && threadIdx.x < 32u && cbase + threadIdx.x < B) {
        const uint32_t c = cbase + threadIdx.x;
        const uint32_t* rw = reinterpret_cast<const uint32_t*>(ep.rows + c);
        mt[0] = rw[9];  // has_mods
        mt[1] = rw[3];  // repetition_penalty
        mt[2] = rw[4];  // presence_penalty
        mt[3] = rw[5];  // frequency_penalty
        const bool two = tile * kTileRows + 32u < ep.V;
        if (ep.hcount) {
            const uint32_t* hw = ep.hbits + (size_t)c * ep.hbw + 2u * tile;
            mt[4] = hw[0];
            if (two) mt[5] = hw[1];
        }
        if (ep.ban) {
            const uint32_t* bw = ep.ban + (size_t)c * ep.ban_stride + 2u * tile;
            mt[6] = bw[0];
            if (two) mt[7] = bw[1];
        }
        if (ep.block_start) {
            const uint32_t* bs = ep.block_start + (size_t)c * (ep.ntile + 1u) + tile;
            mt[8] = bs[0];
            mt[9] = bs[1];
        }
    }

    uint4 wr[PF][2], xr[PF][4];
    uint32_t sr[PF][2];
    auto load = [&](int p, uint32_t g) {
#pragma unroll
        for (int mb = 0; mb < 2; ++mb) sr[p][mb] = buf_load_b32(srs, soff + 128u * (uint32_t)mb, g * 256u);
#pragma unroll
        for (int mb = 0; mb < 2; ++mb) wr[p][mb] = buf_load_b128(wrs, woff + 512u * (uint32_t)mb, g * 2048u);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const v4u t = __builtin_amdgcn_raw_buffer_load_b128(xrs, xoff, g * ncb * 4096u + 1024u * (uint32_t)j, 0);
            xr[p][j] = make_uint4(t.x, t.y, t.z, t.w);
        }
    };
    f16v acc[2];
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[mb][r] = 0.0f;
    // groups past the range are clamped to the last group: loaded, never used
#pragma unroll
    for (int p = 0; p < PF; ++p) load(p, min(g0 + (uint32_t)p, G - 1u));
    for (uint32_t gb = g0; gb < g1; gb += PF) {
#pragma unroll
        for (int p = 0; p < PF; ++p) {
            if (gb + (uint32_t)p < g1) {  // uniform
                SbHalves h[2];
#pragma unroll
                for (int mb = 0; mb < 2; ++mb) h[mb] = unpack_sb16<DENORM>(sr[p][mb]);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
#pragma unroll
                    for (int mb = 0; mb < 2; ++mb) {
                        const h8v a = dequant_word<DENORM>(word_of(wr[p][mb], j), h[mb].s2, h[mb].b2, h[mb].bx, magic);
                        acc[mb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, __builtin_bit_cast(h8v, xr[p][j]), acc[mb], 0, 0, 0);
                    }
                }
                load(p, min(gb + (uint32_t)(p + PF), G - 1u));
            }
        }
    }

    if (ep.meta && threadIdx.x < 32u) {
#pragma unroll
        for (int k = 0; k < 10; ++k) meta[threadIdx.x][k] = mt[k];
    }
    // partial tiles: column l32, four consecutive rows per 16-byte store
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int q = 0; q < 4; ++q)
            *reinterpret_cast<float4*>(&part[wave][l32 * kPartCol + 32u * mb + 8u * q + 4u * hl]) =
                make_float4(acc[mb][4 * q], acc[mb][4 * q + 1], acc[mb][4 * q + 2], acc[mb][4 * q + 3]);
    __syncthreads();
    const uint32_t ncol = min(32u, B - cbase);
    for (uint32_t c = wave; c < ncol; c += (uint32_t)KS) {
        float l = part[0][c * kPartCol + lane];
#pragma unroll
        for (int w = 1; w < KS; ++w) l = l + part[w][c * kPartCol + lane];
        split_column(l, cbase + c, tile, lane, meta[c], ep);
    }
}

// The waves that share a tile, or 0 for the heads of gemm_mfma.hip. Measured on the whole
// turbo_lmhead_logits call (preparation and head, hidden 2816, us, gemm_mfma.hip -> split):
//   tiles x 32-column blocks   65 x 1: 31.9 -> 11.2    256 x 1: 30.7 -> 13.8   512 x 1: 31.9 -> 20.4
//                              65 x 8: 49.8 -> 27.5    256 x 4: 42.2 -> 30.8   512 x 2: 38.0 -> 31.3
// and the other side of the line: 256 x 8 45.4 -> 53.0, 512 x 4 43.6 -> 51.9, 1024 x 1 33.3 -> 33.8
// (a workgroup here dequantises its tile for 32 columns only, which costs more than the idle CUs
// once there are enough tiles). Eight waves per tile up to 256 tiles, where four would leave the
// chip short of waves (65 x 1 with four: 13.3; 501 x 1 with eight: 16.2 against 15.7).
uint32_t mfma_split_waves(const Head& h, int batch) {
    const uint32_t ncb = ((uint32_t)batch + 31u) / 32u;
    if (h.ntile > 768u || h.ntile * ncb > 1024u) return 0u;
    return h.ntile <= 256u ? 8u : 4u;
}

void launch_head_mfma_split(const Head& h, int batch, const EpiArgs& ep, hipStream_t st, hipEvent_t ev0, hipEvent_t ev1) {
    const uint32_t B = (uint32_t)batch, ncb = (B + 31u) / 32u;
    const uint32_t ks = mfma_split_waves(h, batch);
    const dim3 grid(ncb * ((h.ntile + 7u) / 8u) * 8u);
#define TDT_LAUNCH(KS, DN)                                                                                       \
    hipExtLaunchKernelGGL((k_head_mfma_split<KS, DN>), grid, dim3(64 * KS), 0, st, ev0, ev1, 0, h.Wt, h.SB16t, h.x16, B, \
                          h.NC, h.G, ncb, ep)
    if (ks == 8u) {
        if (h.mfma_denorm) TDT_LAUNCH(8, true);
        else TDT_LAUNCH(8, false);
    } else if (ks == 4u) {
        if (h.mfma_denorm) TDT_LAUNCH(4, true);
        else TDT_LAUNCH(4, false);
    } else {
        throw std::runtime_error("split MFMA head: too many tiles");
    }
#undef TDT_LAUNCH
    check_hip(hipGetLastError(), "head (MFMA, split groups)");
}

}  // namespace tdt
