// Small-batch (B <= 2) affine-int4 LM head: a bandwidth-bound streaming GEMV.
//
// Reference semantics: out[row] = sum_g s_g * sum_j q_j x_j + b_g * sum_j x_j
// (src/cpu_reference.cpp:55-84; shaders/GemvInt4.hlsl + Common.hlsli:98-141).
//
// Design (gfx950):
//  * One wave64 per 64-row tile, lane = row. The tiled layout makes each wave's load of one
//    16-byte chunk a contiguous 1 KiB (64 lanes x global_load_dwordx4); a tile is one 88 KiB
//    contiguous stream at D = 2816.
//  * Activations are block floating point with 21-bit mantissas per 64-element group, split
//    into six signed 4-bit digit planes. With q' = q - 8 (one XOR of the word with 0x88888888)
//    every weight word needs six v_dot8_i32_i4 against wave-uniform digit words that live in
//    SGPRs (scalar loads). Products are exact integers, so only the per-group scale-back and
//    the fp32 group combination round:
//        row += s * (D_g * 2^(e-21)) + (8 s + b) * S_g,   D_g = sum q'_j X_j,  S_g = sum X_j 2^(e-21)
//  * Per-group scale/bias come from the tiled (s | b << 16) words, one coalesced dword per lane.
//  * Loads are nontemporal and software-pipelined kPF groups ahead.
#include <hip/hip_ext.h>

#include <algorithm>
#include <stdexcept>
#include <type_traits>

#include "dt_epilogue.h"

namespace tdt {

constexpr int kDigitWaves = 4;
// Groups in flight per wave. With nontemporal loads a shallow pipeline streams fastest: on
// MI355X depth 1-2 reaches 6.6 TB/s where depth 4 (more VGPRs, fewer resident waves) gave
// 6.1 TB/s and plain loads 5.3 TB/s.
constexpr int kPF = 2;

typedef unsigned v4u __attribute__((ext_vector_type(4)));

// The table is streamed once per step: nontemporal loads keep it from displacing the
// activations and partials in the caches.
__device__ inline uint4 load_stream(const uint4* p) {
    const v4u t = __builtin_nontemporal_load(reinterpret_cast<const v4u*>(p));
    return make_uint4(t.x, t.y, t.z, t.w);
}
__device__ inline uint32_t load_stream(const uint32_t* p) { return __builtin_nontemporal_load(p); }

template <int NB>
__global__ __launch_bounds__(kDigitWaves * 64) void k_head_digits(
    const uint4* __restrict__ Wt, const uint32_t* __restrict__ SBt, const uint32_t* __restrict__ xdig,
    const float* __restrict__ xws, const float* __restrict__ xsum, uint32_t NC, uint32_t G, EpiArgs ep) {
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t tile = blockIdx.x * kDigitWaves + wave;
    if (tile >= ep.ntile) return;  // wave-uniform
    const uint4* wp = Wt + (size_t)tile * NC * kTileRows + lane;
    const uint32_t* sbp = SBt + (size_t)tile * G * kTileRows + lane;

    float acc[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[nb] = 0.0f;

    uint4 wa[kPF], wb[kPF];
    uint32_t sb[kPF];
#pragma unroll
    for (int p = 0; p < kPF; ++p) {
        if ((uint32_t)p < G) {
            wa[p] = load_stream(wp + (size_t)(2 * p) * kTileRows);
            wb[p] = load_stream(wp + (size_t)(2 * p + 1) * kTileRows);
            sb[p] = load_stream(sbp + (size_t)p * kTileRows);
        }
    }

    for (uint32_t g0 = 0; g0 < G; g0 += kPF) {
#pragma unroll
        for (int p = 0; p < kPF; ++p) {
            const uint32_t g = g0 + p;
            if (g < G) {
                const uint4 A = wa[p], Bw = wb[p];
                const uint32_t s = sb[p];
                const uint32_t gn = g + kPF;
                if (gn < G) {
                    wa[p] = load_stream(wp + (size_t)(2 * gn) * kTileRows);
                    wb[p] = load_stream(wp + (size_t)(2 * gn + 1) * kTileRows);
                    sb[p] = load_stream(sbp + (size_t)gn * kTileRows);
                }
                const uint32_t wq[8] = {A.x ^ 0x88888888u, A.y ^ 0x88888888u, A.z ^ 0x88888888u,
                                        A.w ^ 0x88888888u, Bw.x ^ 0x88888888u, Bw.y ^ 0x88888888u,
                                        Bw.z ^ 0x88888888u, Bw.w ^ 0x88888888u};
                const float sf = bf16_to_f32(s & 0xFFFFu);
                const float bf = bf16_to_f32(s >> 16);
                const float c8 = fmaf(8.0f, sf, bf);
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) {
                    const uint32_t* xd = xdig + ((size_t)nb * NC + 2u * g) * kDigitWordsPerChunk;
                    int a[kDigits];
#pragma unroll
                    for (uint32_t k = 0; k < kDigits; ++k) a[k] = 0;
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
#pragma unroll
                            for (uint32_t k = 0; k < kDigits; ++k)
                                a[k] = __builtin_amdgcn_sdot8((int)wq[4 * h + i],
                                                              (int)xd[h * kDigitWordsPerChunk + k * 4 + i],
                                                              a[k], false);
                        }
                    }
                    uint32_t Dg = (uint32_t)a[0];
#pragma unroll
                    for (uint32_t k = 1; k < kDigits; ++k) Dg += (uint32_t)a[k] << (4u * k);
                    const float t = sf * xws[(size_t)nb * G + g];
                    acc[nb] = fmaf((float)(int)Dg, t, acc[nb]);
                    acc[nb] = fmaf(c8, xsum[(size_t)nb * G + g], acc[nb]);
                }
            }
        }
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) epilogue_wave(acc[nb], (uint32_t)nb, tile, lane, ep);
}

// ---- the small-batch step with the preparation folded in ------------------------------------
// One workgroup of 16 waves (one per CU) covers 16 consecutive tiles. Before streaming, each
// workgroup recomputes what the step-prep kernel would have written, keeping it in LDS:
//   * final RMSNorm (src/cpu_reference.cpp:43-52): double sum of squares, float mean + eps,
//     1 / sqrt, each correctly rounded;
//   * the block floating-point form of every 64-element group and its six digit planes: thread
//     t owns octet t (elements 8t .. 8t + 7), so a group is 8 lanes (three DPP steps for its
//     maximum and sum) and a lane writes its own digit words, the balanced base-16 digits of
//     X read off Y = X + 0x888888 (its nibbles minus 8);
//   * the occurrence count of each of its own 1024 ids in the row's history
//     (src/sampling.cpp:81-89 visits every occurrence; ids past the vocabulary are ignored).
// The loads of the row, its norm weight and its history are issued first, then the weight
// prefetch, so this work runs while the first groups are in flight; it replaces a kernel launch
// and its dependent-launch gap. Workgroup 0 also copies the row parameters to device memory for
// the select kernel, after its stream.
// The sum of squares adds in a different order from the step-prep kernel; the mean is rounded
// to float from double either way, so the two agree except at a rounding tie of that float.
constexpr uint32_t kFusedWaves = 16;
constexpr uint32_t kFusedThreads = kFusedWaves * 64;
constexpr uint32_t kFusedHistPer = kFusedHistMax / kFusedThreads;
static_assert(kFusedMaxD == 8u * kFusedThreads, "one octet per thread");

template <int NB>
struct FusedLds {
    uint32_t dig[NB][kFusedMaxD / 32 * kDigitWordsPerChunk];
    float ws[NB][kFusedMaxD / 64];
    float sum[NB][kFusedMaxD / 64];
    uint32_t cnt[NB][kFusedThreads];  // history occurrences of the workgroup's ids
    double red[NB][kFusedWaves];
};

// What the preparation reads, loaded before the weight stream is issued (loads complete in
// order, so waiting for these does not wait for the stream).
template <int NB>
struct FusedIn {
    uint4 x[NB][2];  // the thread's octet: fp32 in both, or bf16 pairs in the first
    uint4 gw;        // the octet's bf16 norm weights
    uint32_t hlen[NB];
    uint32_t hid[NB][kFusedHistPer];
};

// Whether row nb's history is counted.
__device__ inline bool fused_hist_on(const FusedPrep& fp, int nb) {
    return fp.history != nullptr && (fp.inl[nb].has_mods & 1u) != 0u;
}

template <int NB, bool HIST = true>
__device__ inline void fused_load(const FusedPrep& fp, uint32_t D, FusedIn<NB>& in) {
    // Every load is unconditional, from an address that is always valid (the octet clamped to the
    // row; an absent input reads the hidden row instead and is ignored), and nothing is done with
    // the loaded bits here: a select or branch on a loaded value would make the wave wait for it.
    const uint32_t tid = threadIdx.x;
    const uint32_t o = min(tid, D / 8u - 1u);
    const uint32_t esz = (fp.dtype == 1) ? 2u : 4u;
    const char* xb = reinterpret_cast<const char*>(fp.hidden);
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        const size_t off = (size_t)esz * ((size_t)nb * D + 8u * o);
        in.x[nb][0] = *reinterpret_cast<const uint4*>(xb + off);
        in.x[nb][1] = *reinterpret_cast<const uint4*>(xb + off + (esz == 4u ? 16u : 0u));
    }
    in.gw = fp.gamma ? reinterpret_cast<const uint4*>(fp.gamma)[o] : *reinterpret_cast<const uint4*>(xb);
    if constexpr (!HIST) return;
    const uint32_t* xw = reinterpret_cast<const uint32_t*>(fp.hidden);
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        const bool on = fused_hist_on(fp, nb);
        const uint32_t* h = on ? fp.history + (size_t)nb * fp.hist_stride : xw;
        const uint32_t lim = on ? fp.hist_stride - 1u : 0u;
        in.hlen[nb] = *(on ? fp.hist_len + nb : xw);
#pragma unroll
        for (uint32_t q = 0; q < kFusedHistPer; ++q) in.hid[nb][q] = h[min(tid + q * kFusedThreads, lim)];
    }
}

__device__ inline uint32_t word_at(const uint4& v, int i) {
    return (i == 0) ? v.x : (i == 1) ? v.y : (i == 2) ? v.z : v.w;
}

// value of 8-lane group reduction (lanes 8k .. 8k + 7)
template <class T, class Op>
__device__ inline T octet_group_reduce(T v, Op op) {
    v = op(v, dpp_mov<dpp::kXor1>(v));
    v = op(v, dpp_mov<dpp::kXor2>(v));
    v = op(v, dpp_mov<dpp::kHalfMirror>(v));
    return v;
}

// HIST: also counts the history of the workgroup's ids, 1024 from blockIdx.x * 1024 on.
template <int NB, bool HIST = true>
__device__ __attribute__((always_inline)) inline void fused_prep(const FusedPrep& fp, uint32_t D, uint32_t V, const FusedIn<NB>& in, FusedLds<NB>& s) {
#pragma clang fp contract(off)
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t idbase = blockIdx.x * kFusedThreads;
    const bool ov = 8u * tid < D;  // this thread's octet lies in the row
    // the octet's elements (0 past the row)
    auto elems = [&](int nb, float (&v)[8]) {
        if (fp.dtype == 1) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t w = word_at(in.x[nb][0], i);
                v[2 * i] = bf16_to_f32(w & 0xFFFFu);
                v[2 * i + 1] = bf16_to_f32(w >> 16);
            }
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = __uint_as_float(word_at(in.x[nb][i >> 2], i & 3));
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = ov ? v[i] : 0.0f;
    };
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        if constexpr (HIST) s.cnt[nb][tid] = 0u;
        if (!fp.normed) {
            float v[8];
            elems(nb, v);
            double acc = 0.0;
#pragma unroll
            for (int i = 0; i < 8; ++i) acc += (double)v[i] * (double)v[i];
            acc = wave_sum_d(acc);
            if (lane == 0) s.red[nb][wave] = acc;
        }
    }
    __syncthreads();  // partial sums written; counts zeroed
    if constexpr (HIST) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        const uint32_t nh = fused_hist_on(fp, nb) ? min(in.hlen[nb], fp.hist_stride) : 0u;
#pragma unroll
        for (uint32_t q = 0; q < kFusedHistPer; ++q) {
            const uint32_t i = tid + q * kFusedThreads, id = in.hid[nb][q];
            if (i < nh && id < V && id - idbase < kFusedThreads) atomicAdd(&s.cnt[nb][id - idbase], 1u);
        }
    }
    }
    const uint32_t g = tid >> 3, j8 = tid & 7u;  // group and octet within it
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        if (8u * 64u * wave >= D) break;  // wave-uniform: no octet of this wave lies in the row
        float v[8];
        elems(nb, v);
        if (!fp.normed) {
            const double tot = wave_sum_d(lane < (blockDim.x >> 6) ? s.red[nb][lane] : 0.0);
            const float ms = (float)(tot / (double)D);
            // sqrtf and 1.0f / s, each correctly rounded: computed in double and rounded once
            const float sq = (float)sqrt((double)(ms + fp.eps));
            const float inv = (float)(1.0 / (double)sq);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                v[i] = v[i] * inv;
                if (fp.gamma) {
                    const uint32_t w = word_at(in.gw, i >> 1);
                    v[i] = v[i] * bf16_to_f32((i & 1) ? (w >> 16) : (w & 0xFFFFu));
                }
            }
        }
        float m = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; ++i) m = fmaxf(m, fabsf(v[i]));
        m = octet_group_reduce(m, [](float a, float b) { return fmaxf(a, b); });
        int e = 0;
        (void)frexpf(m, &e);  // m = f * 2^e, f in [0.5, 1); e = 0 for m = 0
        int X[8], sX = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            X[i] = (int)rintf(ldexpf(v[i], 21 - e));
            sX += X[i];
        }
        sX = octet_group_reduce(sX, [](int a, int b) { return a + b; });
        if (ov && j8 == 0u) {
            s.ws[nb][g] = ldexpf(1.0f, e - 21);
            s.sum[nb][g] = (float)sX * ldexpf(1.0f, e - 21);
        }
        uint32_t Z[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) Z[i] = ((uint32_t)X[i] + 0x888888u) ^ 0x888888u;
        uint32_t* dst = &s.dig[nb][(2u * g + (j8 >> 2)) * kDigitWordsPerChunk + (j8 & 3u)];
#pragma unroll
        for (uint32_t k = 0; k < kDigits; ++k) {
            uint32_t w = 0u;
#pragma unroll
            for (int i = 0; i < 8; ++i) w |= ((Z[i] >> (4u * k)) & 15u) << (4u * i);
            if (ov) dst[k * 4u] = w;
        }
    }
    __syncthreads();  // digits, scales and counts complete
}

template <int NB>
__global__ __launch_bounds__(kFusedThreads) void k_head_digits_fused(
    const uint4* __restrict__ Wt, const uint32_t* __restrict__ SBt, uint32_t D, uint32_t NC, uint32_t G,
    FusedPrep fp, EpiArgs ep) {
    __shared__ __attribute__((aligned(16))) FusedLds<NB> s;
    const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t tile_raw = blockIdx.x * kFusedWaves + wave;
    const bool tile_ok = tile_raw < ep.ntile;
    const uint32_t tile = tile_ok ? tile_raw : ep.ntile - 1u;  // loads clamped; no epilogue
    const uint4* wp = Wt + (size_t)tile * NC * kTileRows + lane;
    const uint32_t* sbp = SBt + (size_t)tile * G * kTileRows + lane;

    FusedIn<NB> in;
    fused_load<NB>(fp, D, in);
    __builtin_amdgcn_sched_barrier(0);  // keep the row's loads ahead of the weight stream
    // branch-free (a group past the end is a repeated, unused load): with a branch here the
    // compiler's wait for the row's loads would have to assume the shorter path and also wait
    // for part of the stream
    uint4 wa[kPF], wb[kPF];
    uint32_t sb[kPF];
#pragma unroll
    for (int p = 0; p < kPF; ++p) {
        const uint32_t gp = min((uint32_t)p, G - 1u);
        wa[p] = load_stream(wp + (size_t)(2 * gp) * kTileRows);
        wb[p] = load_stream(wp + (size_t)(2 * gp + 1) * kTileRows);
        sb[p] = load_stream(sbp + (size_t)gp * kTileRows);
    }
    __builtin_amdgcn_sched_barrier(0);
    fused_prep<NB>(fp, D, ep.V, in, s);

    float acc[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[nb] = 0.0f;
    for (uint32_t g0 = 0; g0 < G; g0 += kPF) {
#pragma unroll
        for (int p = 0; p < kPF; ++p) {
            const uint32_t g = g0 + p;
            if (g < G) {
                const uint4 A = wa[p], Bw = wb[p];
                const uint32_t sbw = sb[p];
                const uint32_t gn = g + kPF;
                if (gn < G) {
                    wa[p] = load_stream(wp + (size_t)(2 * gn) * kTileRows);
                    wb[p] = load_stream(wp + (size_t)(2 * gn + 1) * kTileRows);
                    sb[p] = load_stream(sbp + (size_t)gn * kTileRows);
                }
                const uint32_t wq[8] = {A.x ^ 0x88888888u, A.y ^ 0x88888888u, A.z ^ 0x88888888u,
                                        A.w ^ 0x88888888u, Bw.x ^ 0x88888888u, Bw.y ^ 0x88888888u,
                                        Bw.z ^ 0x88888888u, Bw.w ^ 0x88888888u};
                const float sf = bf16_to_f32(sbw & 0xFFFFu);
                const float bf = bf16_to_f32(sbw >> 16);
                const float c8 = fmaf(8.0f, sf, bf);
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) {
                    const uint32_t* xd = &s.dig[nb][(2u * g) * kDigitWordsPerChunk];
                    int a[kDigits];
#pragma unroll
                    for (uint32_t k = 0; k < kDigits; ++k) a[k] = 0;
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
#pragma unroll
                            for (uint32_t k = 0; k < kDigits; ++k)
                                a[k] = __builtin_amdgcn_sdot8((int)wq[4 * h + i],
                                                              (int)xd[h * kDigitWordsPerChunk + k * 4 + i],
                                                              a[k], false);
                        }
                    }
                    uint32_t Dg = (uint32_t)a[0];
#pragma unroll
                    for (uint32_t k = 1; k < kDigits; ++k) Dg += (uint32_t)a[k] << (4u * k);
                    const float t = sf * s.ws[nb][g];
                    acc[nb] = fmaf((float)(int)Dg, t, acc[nb]);
                    acc[nb] = fmaf(c8, s.sum[nb][g], acc[nb]);
                }
            }
        }
    }
    // the row parameters for the select kernel (after the stream: this wait is free here)
    if (blockIdx.x == 0u && threadIdx.x < NB * (sizeof(DevRow) / 4))
        reinterpret_cast<uint32_t*>(fp.rows_dst)[threadIdx.x] = reinterpret_cast<const uint32_t*>(&fp.inl[0])[threadIdx.x];
    if (!tile_ok) return;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        const uint32_t cnt = (fp.inl[nb].has_mods & 1u) ? s.cnt[nb][wave * 64u + lane] : 0u;
        epilogue_wave_counted(acc[nb], (uint32_t)nb, tile, lane, ep, fp.inl[nb], cnt);
    }
}

void launch_head_small(const Head& h, int batch, const FusedPrep* fp, const EpiArgs& ep, hipStream_t st, hipEvent_t ev0,
                       hipEvent_t ev1);

void launch_head_digits_fused(const Head& h, int batch, const FusedPrep& fp, const EpiArgs& ep,
                              hipStream_t st, hipEvent_t ev0, hipEvent_t ev1) {
    if (h.D > kFusedMaxD || h.D % kGroup != 0u) throw std::runtime_error("folded step needs D <= 8192");
    if (h.ntile < kFusedMinTiles) {
        launch_head_small(h, batch, &fp, ep, st, ev0, ev1);
        return;
    }
    const dim3 grid((h.ntile + kFusedWaves - 1u) / kFusedWaves), block(kFusedThreads);
    if (batch == 1)
        hipExtLaunchKernelGGL(k_head_digits_fused<1>, grid, block, 0, st, ev0, ev1, 0, h.Wt, h.SBt, h.D, h.NC,
                              h.G, fp, ep);
    else if (batch == 2)
        hipExtLaunchKernelGGL(k_head_digits_fused<2>, grid, block, 0, st, ev0, ev1, 0, h.Wt, h.SBt, h.D, h.NC,
                              h.G, fp, ep);
    else
        throw std::runtime_error("folded step supports batch 1 or 2");
    check_hip(hipGetLastError(), "head (digit GEMV, folded preparation)");
}

constexpr uint32_t kMaxSplit = 16;  // waves of a workgroup that shares a tile

// Waves per workgroup, from the row's length alone: eight, fewer where the row has fewer units, more
// where a thread per 8 elements needs them. Sixteen repeat more preparation (704 x 2816: 4.1 us a call
// with four, 4.1 with eight, 4.9 with sixteen; 65,536 x 1600: 10.4, 10.7, 12.3).
inline uint32_t mv_waves(uint32_t D) { return std::max(std::min(8u, (D / 32u + 3u) / 4u), (D / 8u + 63u) / 64u); }

// Two rows over 1025 .. 2047 tiles: two or four waves to a tile, with the digit words of the preparation
// kernel in scalar registers. Enough tiles fill the chip, and k_head_small's digit reads through LDS,
// two rows' worth for every chunk, cost more than the launch it saves. Whole sampled step, us, here and
// with k_head_small: 131,000 x 2816 52.8 and 61.5; at the line the launch weighs as much as the reads:
// 65,536 x 512 21.9 and 19.4, x 1600 28.3 and 29.5, x 2816 36.3 and 39.9.
// The sums are k_head_small's, so a row's logits do not depend on the row beside it: the same ranges of
// units of two groups (mv_waves of them, here split over the two waves), an accumulator to each place in
// a unit, and the ranges added in order.
bool digits_pair(const Head& h, int batch) { return batch == 2 && h.ntile > 1024u && h.ntile < kFusedMinTiles; }

// PW: the waves of a workgroup, four where a range holds more than a unit (sampled steps, us with two /
// four: 66,000 x 768 27.2 / 22.7, 98,304 x 2816 53.8 / 42.6, 131,000 x 2816 57.8 / 52.8; but 98,304 x
// 512 24.0 / 26.1).
constexpr uint32_t kPairFourD = 768;
// inv: 2^16 / KS rounded up, which divides a range's first unit exactly (x inv >> 16 for x = r U <= 16 x 64).
template <uint32_t PW>
__global__ __launch_bounds__(64 * PW) void k_head_digits_pair(
    const uint4* __restrict__ Wt, const uint32_t* __restrict__ SBt, const uint32_t* __restrict__ xdig,
    const float* __restrict__ xws, const float* __restrict__ xsum, uint32_t NC, uint32_t G, uint32_t KS, uint32_t inv,
    EpiArgs ep) {
    constexpr int NB = 2;
    __shared__ float part[kMaxSplit][NB][64];  // by range
    // wave-uniform by construction; read through the scalar unit so the group range, and with it
    // the digit-word addresses, stay scalar (s_load) instead of per-lane loads
    const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t tile = blockIdx.x, U = (NC + 3u) / 4u;
    const uint4* wp = Wt + (size_t)tile * NC * kTileRows + lane;
    const uint32_t* sbp = SBt + (size_t)tile * G * kTileRows + lane;
    float acc[NB][2] = {};
    auto first_unit = [&](uint32_t range) { return (range * U * inv) >> 16; };  // range U / KS
    uint32_t r = wave * KS / PW;  // the wave's current range, and the unit it ends before
    const uint32_t r1 = (wave + 1u) * KS / PW;
    uint32_t uend = first_unit(r + 1u);
    const uint32_t g0 = 2u * first_unit(r), g1 = min(2u * first_unit(r1), G);  // a unit is two groups
    // all of a batch of kBatchG groups are loaded before any is used, so the wave waits for memory
    // once per batch rather than once per group
    constexpr uint32_t kBatchG = 4;
    for (uint32_t gb = g0; gb < g1; gb += kBatchG) {
        uint4 Ab[kBatchG], Bb[kBatchG];
        uint32_t Sb[kBatchG];
#pragma unroll
        for (uint32_t q = 0; q < kBatchG; ++q) {
            const uint32_t g = min(gb + q, g1 - 1u);  // past the range: a repeated, unused load
            Ab[q] = load_stream(wp + (size_t)(2 * g) * kTileRows);
            Bb[q] = load_stream(wp + (size_t)(2 * g + 1) * kTileRows);
            Sb[q] = load_stream(sbp + (size_t)g * kTileRows);
        }
#pragma unroll
        for (uint32_t q = 0; q < kBatchG; ++q) {
            // branch-free: a group past the range is computed on its clamped copy and dropped,
            // so no branch separates the batch's loads from each other
            const bool in = gb + q < g1;
            const uint32_t g = min(gb + q, g1 - 1u);
            const uint4 A = Ab[q], Bw = Bb[q];
            const uint32_t wq[8] = {A.x ^ 0x88888888u, A.y ^ 0x88888888u, A.z ^ 0x88888888u,
                                    A.w ^ 0x88888888u, Bw.x ^ 0x88888888u, Bw.y ^ 0x88888888u,
                                    Bw.z ^ 0x88888888u, Bw.w ^ 0x88888888u};
            const float sf = bf16_to_f32(Sb[q] & 0xFFFFu);
            const float bf = bf16_to_f32(Sb[q] >> 16);
            const float c8 = fmaf(8.0f, sf, bf);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                const uint32_t* xd = xdig + ((size_t)nb * NC + 2u * g) * kDigitWordsPerChunk;
                int a[kDigits];
#pragma unroll
                for (uint32_t k = 0; k < kDigits; ++k) a[k] = 0;
#pragma unroll
                for (int hh = 0; hh < 2; ++hh)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
#pragma unroll
                        for (uint32_t k = 0; k < kDigits; ++k)
                            a[k] = __builtin_amdgcn_sdot8((int)wq[4 * hh + i],
                                                          (int)xd[hh * kDigitWordsPerChunk + k * 4 + i], a[k], false);
                uint32_t Dg = (uint32_t)a[0];
#pragma unroll
                for (uint32_t k = 1; k < kDigits; ++k) Dg += (uint32_t)a[k] << (4u * k);
                float& s = acc[nb][q & 1u];  // g0 and the batches are even: q & 1 = g & 1
                float t = fmaf((float)(int)Dg, sf * xws[(size_t)nb * G + g], s);
                t = fmaf(c8, xsum[(size_t)nb * G + g], t);
                s = in ? t : s;
            }
            if ((q & 1u) && ((gb + q) >> 1) + 1u == uend) {  // uniform: the range's last unit
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) {
                    part[r][nb][lane] = acc[nb][0] + acc[nb][1];
                    acc[nb][0] = acc[nb][1] = 0.0f;
                }
                ++r;
                uend = (r < r1) ? first_unit(r + 1u) : 0u;
            }
        }
    }
    __syncthreads();
    if (wave >= (uint32_t)NB) return;
    // wave nb adds row nb's ranges and runs its epilogue
    float v = part[0][wave][lane];
    for (uint32_t w = 1; w < KS; ++w) v += part[w][wave][lane];
    epilogue_wave(v, wave, tile, lane, ep);
}

void launch_head_digits(const Head& h, int batch, const EpiArgs& ep, hipStream_t st,
                        hipEvent_t ev0, hipEvent_t ev1) {
    if (digits_pair(h, batch)) {
        const uint32_t pw = h.D >= kPairFourD ? 4u : 2u, ks = mv_waves(h.D), inv = (65536u + ks - 1u) / ks;
        hipExtLaunchKernelGGL(pw == 4u ? k_head_digits_pair<4> : k_head_digits_pair<2>, dim3(h.ntile), dim3(64u * pw), 0, st,
                              ev0, ev1, 0, h.Wt, h.SBt, h.xdig, h.xws, h.xsum, h.NC, h.G, ks, inv, ep);
        check_hip(hipGetLastError(), "head (digit GEMV, two rows, wave pairs)");
        return;
    }
    if (h.ntile < kFusedMinTiles) {
        launch_head_small(h, batch, nullptr, ep, st, ev0, ev1);
        return;
    }
    const unsigned grid = (h.ntile + kDigitWaves - 1) / kDigitWaves;
    if (batch == 1)
        hipExtLaunchKernelGGL(k_head_digits<1>, dim3(grid), dim3(kDigitWaves * 64), 0, st, ev0, ev1,
                              0, h.Wt, h.SBt, h.xdig, h.xws, h.xsum, h.NC, h.G, ep);
    else if (batch == 2)
        hipExtLaunchKernelGGL(k_head_digits<2>, dim3(grid), dim3(kDigitWaves * 64), 0, st, ev0, ev1,
                              0, h.Wt, h.SBt, h.xdig, h.xws, h.xsum, h.NC, h.G, ep);
    else
        throw std::runtime_error("digit GEMV supports batch 1 or 2");
    check_hip(hipGetLastError(), "head (digit GEMV)");
}

// ---- matrix-vector products: raw outputs of one or two rows, and of several matrices at once -------
// A projection's product is a few microseconds of launch, round trips and one compute unit's issue
// rate, not bandwidth, so a tile's 64 rows are divided among Q workgroups: in a wave, 64 / Q rows times
// Q slots of chunks of 32 elements (lane = row + (64 / Q) * slot). Chunks come in units of four, two
// 64-element groups, split over KS waves; a lane takes 4 / Q consecutive chunks of each unit. A group's
// integer sum is formed whole (over two lanes at Q = 4) and goes into the accumulator of its place in
// the unit, so that the sums (per wave and place, then over the two places, then over the waves in
// order) are the same for every Q and round once per group. Each workgroup computes the digit planes
// of the whole row into LDS (fused_prep) while its first weights load. Needs one thread per 8 elements.
template <int NB>
struct MvLds {
    float part[2][kMaxSplit][NB][64];  // by the parity of the workgroup's tile
    FusedLds<NB> f;
};

// Workgroups per tile, from the tiles of the launch. A call of one matrix, us at Q = 1 / 2 / 4 (one
// wave per whole tile, which this replaced, in brackets):
//   704 x 2816 (11 tiles)   5.78  5.09  4.08  [7.44]     8192 x 2816 (128)   6.47  5.49  5.65  [8.28]
//   4096 x 2816 (64)        6.29  5.41  4.17  [7.62]     16384 x 2816 (256)  6.52  6.98  8.15  [8.21]
// A grouped launch's kernel, us: 16 of 704 x 2816 (176 tiles) 7.7  8.5  8.7; 8 of 2816 x 704 (352)
// 5.6  5.9  7.8.
inline uint32_t mv_parts(uint32_t tiles) { return (tiles <= 64u) ? 4u : (tiles <= 128u) ? 2u : 1u; }

// A lane's view of a tile: its row, chunk slot and the wave's units, with the first batch of weights.
template <int Q>
struct MvLane {
    static constexpr uint32_t kRows = 64u / Q, kT = 4u / Q;  // rows of a wave; chunks of a unit to a lane
    static constexpr uint32_t kUnits = Q;                    // units loaded ahead of their use: four chunks
    static constexpr uint32_t kS = (kT + 1u) / 2u;           // groups of a unit to a lane (at Q = 4 half of one)
    uint32_t G, NC, r, slot, u0, u1;
    uint4 W[kUnits][kT];
    uint32_t S[kUnits][kS];
    __device__ __attribute__((always_inline)) MvLane(uint32_t D, uint32_t KS, uint32_t part) {
        const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        G = D / kGroup;
        NC = D / 32u;
        const uint32_t U = (NC + 3u) / 4u;
        r = part * kRows + (lane & (kRows - 1u));
        slot = lane / kRows;
        u0 = (wave < KS) ? wave * U / KS : 0u;
        u1 = (wave < KS) ? (wave + 1u) * U / KS : 0u;
    }
    __device__ __attribute__((always_inline)) void load(const uint4* Wt, const uint32_t* SBt, uint32_t tile, uint32_t ub) {
        const uint4* wp = Wt + (size_t)tile * NC * kTileRows + r;
        const uint32_t* sbp = SBt + (size_t)tile * G * kTileRows + r;
#pragma unroll
        for (uint32_t q = 0; q < kUnits; ++q)
#pragma unroll
            for (uint32_t t = 0; t < kT; ++t) {
                const uint32_t c = min((ub + q) * 4u + kT * slot + t, NC - 1u);  // past the row: repeated, unused
                W[q][t] = load_stream(wp + (size_t)c * kTileRows);
                if (t % 2u == 0u) S[q][t / 2u] = load_stream(sbp + (size_t)(c >> 1) * kTileRows);
            }
    }
};

// The wave's partial sums of a tile whose first batch is loaded, into part (MvLds::part of the tile).
template <int NB, int Q>
__device__ __attribute__((always_inline)) inline void mv_dots(MvLane<Q>& L, const uint4* Wt, const uint32_t* SBt, uint32_t tile,
                                                              const FusedLds<NB>& f, float (&part)[kMaxSplit][NB][64]) {
    constexpr uint32_t kT = MvLane<Q>::kT, kUnits = MvLane<Q>::kUnits, kS = MvLane<Q>::kS;
    constexpr uint32_t kC = kT / kS;  // chunks of a group to a lane
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    float acc[NB][kS];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (uint32_t p = 0; p < kS; ++p) acc[nb][p] = 0.0f;
    for (uint32_t ub = L.u0; ub < L.u1; ub += kUnits) {
        if (ub != L.u0) L.load(Wt, SBt, tile, ub);
#pragma unroll
        for (uint32_t q = 0; q < kUnits; ++q) {
            if (ub + q < L.u1) {  // uniform
#pragma unroll
                for (uint32_t p = 0; p < kS; ++p) {
                    const uint32_t cr = (ub + q) * 4u + kT * L.slot + kC * p, g = min(cr >> 1, L.G - 1u);
                    uint32_t wq[kC][4];
#pragma unroll
                    for (uint32_t t = 0; t < kC; ++t) {
                        const uint4 w = L.W[q][kC * p + t];
                        wq[t][0] = w.x ^ 0x88888888u;
                        wq[t][1] = w.y ^ 0x88888888u;
                        wq[t][2] = w.z ^ 0x88888888u;
                        wq[t][3] = w.w ^ 0x88888888u;
                    }
                    const float sf = bf16_to_f32(L.S[q][p] & 0xFFFFu);
                    const float bf = bf16_to_f32(L.S[q][p] >> 16);
                    const float c8 = fmaf(8.0f, sf, bf);
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb) {
                        uint32_t Dg = 0u;
#pragma unroll
                        for (uint32_t k = 0; k < kDigits; ++k) {
                            int d = 0;
#pragma unroll
                            for (uint32_t t = 0; t < kC; ++t) {
                                const uint32_t c = min(cr + t, L.NC - 1u);
                                const uint4 x = reinterpret_cast<const uint4*>(&f.dig[nb][c * kDigitWordsPerChunk])[k];
                                d = __builtin_amdgcn_sdot8((int)wq[t][0], (int)x.x, d, false);
                                d = __builtin_amdgcn_sdot8((int)wq[t][1], (int)x.y, d, false);
                                d = __builtin_amdgcn_sdot8((int)wq[t][2], (int)x.z, d, false);
                                d = __builtin_amdgcn_sdot8((int)wq[t][3], (int)x.w, d, false);
                            }
                            Dg += (uint32_t)d << (4u * k);
                        }
                        if constexpr (kC == 1u) Dg = sum_xor16(Dg);  // the group's other chunk: the next slot
                        float v = fmaf((float)(int)Dg, sf * f.ws[nb][g], acc[nb][p]);
                        v = fmaf(c8, f.sum[nb][g], v);
                        acc[nb][p] = (cr < L.NC) ? v : acc[nb][p];
                    }
                }
            }
        }
    }
    // over the two places of a unit
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        if constexpr (kS == 2u) part[wave][nb][lane] = acc[nb][0] + acc[nb][1];
        else part[wave][nb][lane] = acc[nb][0] + xor32(acc[nb][0]);
    }
}

// The sum of row nb's partials in wave order, by one wave: lane's row, the same in every slot.
template <int NB>
__device__ __attribute__((always_inline)) inline float mv_sum(const float (&part)[kMaxSplit][NB][64], uint32_t KS, int nb) {
    const uint32_t lane = threadIdx.x & 63u;
    float v = part[0][nb][lane];
    for (uint32_t w = 1; w < KS; ++w) v += part[w][nb][lane];
    return v;
}

// A workgroup's partial sums of one tile part, complete in s.part[0] after its last barrier.
template <int NB, int Q>
__device__ __attribute__((always_inline)) inline void mv_tile(const uint4* Wt, const uint32_t* SBt, uint32_t D, uint32_t KS,
                                                               uint32_t tile, uint32_t part, const FusedPrep& fp,
                                                               MvLds<NB>& s) {
    MvLane<Q> L(D, KS, part);
    FusedIn<NB> in;
    fused_load<NB, false>(fp, D, in);
    __builtin_amdgcn_sched_barrier(0);  // the row's loads ahead of the weights
    L.load(Wt, SBt, tile, L.u0);
    __builtin_amdgcn_sched_barrier(0);
    fused_prep<NB, false>(fp, D, 0u, in, s.f);
    mv_dots<NB, Q>(L, Wt, SBt, tile, s.f, s.part[0]);
    __syncthreads();
}

// The step and greedy heads of one or two rows over fewer than kFusedMinTiles tiles, with the same sums
// as k_matvec: whole tiles (Q = 1), T consecutive ones to a workgroup, the head epilogue by wave nb for
// row nb while the other waves go on to the next tile. FUSED folds the preparation in as the big head
// does (RMSNorm, digit planes, history counts of the workgroup's ids); otherwise the digit planes come
// from the preparation kernel.
template <int NB, bool FUSED>
__global__ __launch_bounds__(kMaxSplit * 64) void k_head_small(const uint4* __restrict__ Wt, const uint32_t* __restrict__ SBt,
                                                               const uint32_t* __restrict__ xdig, const float* __restrict__ xws,
                                                               const float* __restrict__ xsum, uint32_t D, uint32_t T,
                                                               FusedPrep fp, EpiArgs ep) {
    __shared__ __attribute__((aligned(16))) MvLds<NB> s;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t KS = blockDim.x >> 6, t0 = blockIdx.x * T, t1 = min(t0 + T, ep.ntile);
    MvLane<1> L(D, KS, 0u);
    if constexpr (FUSED) {
        FusedIn<NB> in;
        fused_load<NB, false>(fp, D, in);
        __builtin_amdgcn_sched_barrier(0);  // the row's loads ahead of the weights
        L.load(Wt, SBt, t0, L.u0);
        __builtin_amdgcn_sched_barrier(0);
        for (uint32_t i = tid; i < T * kTileRows; i += blockDim.x)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) s.f.cnt[nb][i] = 0u;
        fused_prep<NB, false>(fp, D, ep.V, in, s.f);
        const uint32_t idbase = t0 * kTileRows;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
            if (fused_hist_on(fp, nb)) {
                const uint32_t nh = min(fp.hist_len[nb], fp.hist_stride);
                for (uint32_t i = tid; i < nh; i += blockDim.x) {
                    const uint32_t id = fp.history[(size_t)nb * fp.hist_stride + i];
                    if (id < ep.V && id - idbase < T * kTileRows) atomicAdd(&s.f.cnt[nb][id - idbase], 1u);
                }
            }
    } else {
        L.load(Wt, SBt, t0, L.u0);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            const uint32_t nd = L.NC * kDigitWordsPerChunk;
            for (uint32_t i = tid; i < nd; i += blockDim.x) s.f.dig[nb][i] = xdig[(size_t)nb * nd + i];
            for (uint32_t i = tid; i < L.G; i += blockDim.x) {
                s.f.ws[nb][i] = xws[(size_t)nb * L.G + i];
                s.f.sum[nb][i] = xsum[(size_t)nb * L.G + i];
            }
        }
        __syncthreads();
    }
    for (uint32_t tile = t0; tile < t1; ++tile) {
        auto& part = s.part[(tile - t0) & 1u];  // the other half may still be read by the last epilogue
        mv_dots<NB, 1>(L, Wt, SBt, tile, s.f, part);
        if (tile + 1u < t1) L.load(Wt, SBt, tile + 1u, L.u0);
        __syncthreads();
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            if (wave != (uint32_t)nb % KS) continue;
            const float v = mv_sum<NB>(part, KS, nb);
            if constexpr (FUSED) {
                const uint32_t cnt = (fp.inl[nb].has_mods & 1u) ? s.f.cnt[nb][(tile - t0) * kTileRows + lane] : 0u;
                epilogue_wave_counted(v, (uint32_t)nb, tile, lane, ep, fp.inl[nb], cnt);
            } else {
                epilogue_wave(v, (uint32_t)nb, tile, lane, ep);
            }
        }
    }
    // the row parameters for the select kernel
    if constexpr (FUSED) {
        if (blockIdx.x == 0u && fp.rows_dst)
            for (uint32_t i = tid; i < NB * (sizeof(DevRow) / 4); i += blockDim.x)
                reinterpret_cast<uint32_t*>(fp.rows_dst)[i] = reinterpret_cast<const uint32_t*>(&fp.inl[0])[i];
    }
}

void launch_head_small(const Head& h, int batch, const FusedPrep* fp, const EpiArgs& ep, hipStream_t st, hipEvent_t ev0,
                       hipEvent_t ev1) {
    // Tiles per workgroup, whose preparation they share. The whole sampled step with one row, us, T = 1 /
    // 2 / 4: 32,768 x 2816 (512 tiles) 19.7 20.6 27.5; 65,536 x 2816 30.0 26.6 29.1; 98,304 x 2816 40.0
    // 37.1 37.2; 120,000 x 1600 36.2 31.1 28.7.
    const uint32_t T = (h.ntile > 1536u) ? 4u : (h.ntile > 768u) ? 2u : 1u;
    const dim3 grid((h.ntile + T - 1u) / T), block(64u * mv_waves(h.D));
    const FusedPrep none{};
#define TDT_LAUNCH(NB, F)                                                                                       \
    hipExtLaunchKernelGGL((k_head_small<NB, F>), grid, block, 0, st, ev0, ev1, 0, h.Wt, h.SBt, h.xdig, h.xws, h.xsum, h.D, \
                          T, fp ? *fp : none, ep)
    if (batch == 1) {
        if (fp) TDT_LAUNCH(1, true);
        else TDT_LAUNCH(1, false);
    } else if (batch == 2) {
        if (fp) TDT_LAUNCH(2, true);
        else TDT_LAUNCH(2, false);
    } else {
        throw std::runtime_error("digit GEMV supports batch 1 or 2");
    }
#undef TDT_LAUNCH
    check_hip(hipGetLastError(), "head (digit GEMV, few tiles)");
}

// Logits-only calls of few tiles (with two rows past 1024 tiles the preparation runs on its own and
// k_head_digits_pair serves the call).
bool matvec_small(const Head& h, int batch) { return batch <= kFusedRows && h.ntile < kFusedMinTiles; }

// One or two rows through one matrix (turbo_int4_matvec, turbo_lmhead_logits): softcap, logits only.
template <int NB, int Q>
__global__ __launch_bounds__(kMaxSplit * 64) void k_matvec(const uint4* __restrict__ Wt, const uint32_t* __restrict__ SBt,
                                                           uint32_t D, float* __restrict__ logits, uint32_t V, float cap,
                                                           FusedPrep fp) {
#pragma clang fp contract(off)
    __shared__ __attribute__((aligned(16))) MvLds<NB> s;
    constexpr uint32_t kRows = 64u / Q;
    const uint32_t tile = blockIdx.x / Q, part = blockIdx.x % Q;
    mv_tile<NB, Q>(Wt, SBt, D, blockDim.x >> 6, tile, part, fp, s);
    if (threadIdx.x >= 64u) return;
    const uint32_t id = tile * kTileRows + part * kRows + threadIdx.x;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        float l = mv_sum<NB>(s.part[0], blockDim.x >> 6, nb);
        if (threadIdx.x >= kRows || id >= V) continue;
        if (cap > 0.0f) l = cap * tanhf(l / cap);
        logits[(size_t)nb * V + id] = l;
    }
}

void launch_matvec(const Head& h, int batch, const FusedPrep& fp, const EpiArgs& ep, hipStream_t st, hipEvent_t ev0,
                   hipEvent_t ev1) {
    const uint32_t Q = mv_parts(h.ntile);
    const dim3 grid(h.ntile * Q), block(64u * mv_waves(h.D));
    if (batch != 1 && batch != 2) throw std::runtime_error("matrix-vector product supports batch 1 or 2");
#define TDT_LAUNCH(NB, QQ) \
    hipExtLaunchKernelGGL((k_matvec<NB, QQ>), grid, block, 0, st, ev0, ev1, 0, h.Wt, h.SBt, h.D, ep.logits, h.V, ep.cap, fp)
    if (batch == 1) {
        if (Q == 4u) TDT_LAUNCH(1, 4);
        else if (Q == 2u) TDT_LAUNCH(1, 2);
        else TDT_LAUNCH(1, 1);
    } else {
        if (Q == 4u) TDT_LAUNCH(2, 4);
        else if (Q == 2u) TDT_LAUNCH(2, 2);
        else TDT_LAUNCH(2, 1);
    }
#undef TDT_LAUNCH
    check_hip(hipGetLastError(), "int4 matvec");
}

// Several independent matrices, each with its own input row and output, in one launch: the
// projections a token makes in one layer (the routed experts' gate and up matrices, or their down
// matrices). Workgroup i serves the matrix whose range of tile parts holds i; each output is
// bit-identical to the matrix's own call.
template <int Q>
__global__ __launch_bounds__(kMaxSplit * 64) void k_matvec_grouped(GroupArgs a) {
    __shared__ __attribute__((aligned(16))) MvLds<1> s;
    constexpr uint32_t kRows = 64u / Q;
    // the range starts of all matrices in one load, one to a lane
    const uint32_t lane = threadIdx.x & 63u, wt = blockIdx.x / Q, part = blockIdx.x % Q;
    const uint32_t mi = __builtin_amdgcn_readfirstlane(
        __popcll(__ballot(lane < a.count && wt >= a.tile_begin[min(lane, kMaxGroupMats - 1u)])) - 1u);
    const GroupMat M = a.m[mi];
    const uint32_t tile = wt - a.tile_begin[mi];
    FusedPrep fp{};
    fp.hidden = M.x;
    fp.dtype = 0;
    fp.normed = 1;
    mv_tile<1, Q>(M.Wt, M.SBt, M.D, M.ks, tile, part, fp, s);
    if (threadIdx.x >= 64u) return;
    const float v = mv_sum<1>(s.part[0], M.ks, 0);
    const uint32_t row = tile * kTileRows + part * kRows + threadIdx.x;
    if (threadIdx.x < kRows && row < M.rows) M.out[row] = v;
}

void launch_matvec_grouped(GroupArgs& a, uint32_t tiles, hipStream_t st) {
    if (a.count == 0u) return;
    uint32_t ks = 1u;
    for (uint32_t i = 0; i < a.count; ++i) {
        a.m[i].ks = mv_waves(a.m[i].D);
        ks = std::max(ks, a.m[i].ks);
    }
    const uint32_t Q = mv_parts(tiles);
    const dim3 grid(tiles * Q), block(64u * ks);
    if (Q == 4u) hipLaunchKernelGGL(k_matvec_grouped<4>, grid, block, 0, st, a);
    else if (Q == 2u) hipLaunchKernelGGL(k_matvec_grouped<2>, grid, block, 0, st, a);
    else hipLaunchKernelGGL(k_matvec_grouped<1>, grid, block, 0, st, a);
    check_hip(hipGetLastError(), "grouped int4 matvec");
}

// ---- epilogue over caller-provided logits (no softcap, no GEMV) ----------------------------------
// A wave takes four consecutive tiles of one row, a lane four consecutive ids (one 16-byte load), so
// the block statistics are 16-lane reductions that serve four tiles at once; with one id to a lane
// each 256 bytes of logits paid for its own five 64-lane reductions (16 rows of 262,144 with a ban
// mask: 17.1 us, now 6.5). Logits are stored only where a modifier or the ban changed one.
// Without a preparation kernel (rc.dst) the first workgroups, one per row in the order of the grid, also
// copy the row parameters to device memory for the select kernel: a lane to a word, loaded behind the
// logits and stored at the end, so that the round trip to the staging slot in host memory hides behind
// the rest of the grid. One workgroup for all rows took 14 such round trips at 256 rows (256 x 4096
// 18.0 us, now 4.1); copied by a row's own first workgroup, the last rows' trips came at the end (64 x
// 262,144 sampled 28.2 us a call, now 25.5).
constexpr uint32_t kEpiWaves = 4, kEpiTiles = 4u * kEpiWaves;  // of a workgroup
template <class T, class Op>
__device__ inline T row16_reduce(T v, Op op) {
    v = op(v, dpp_mov<dpp::kXor1>(v));
    v = op(v, dpp_mov<dpp::kXor2>(v));
    v = op(v, dpp_mov<dpp::kRor4>(v));
    return op(v, dpp_mov<dpp::kRor8>(v));
}

__global__ __launch_bounds__(64 * kEpiWaves) void k_logits_epilogue(EpiArgs ep, RowCopy rc, uint32_t mods) {
#pragma clang fp contract(off)
    constexpr uint32_t kRowWords = sizeof(DevRow) / 4u;
    static_assert(kRowWords <= 64u, "one wave copies a row");
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, b = blockIdx.y;
    const uint32_t tile = (blockIdx.x * kEpiWaves + wave) * 4u + (lane >> 4);
    const uint32_t id = tile * kTileRows + 4u * (lane & 15u);  // the lane's first id
    float* lrow = ep.logits + (size_t)b * ep.V;
    const bool vec = (ep.V & 3u) == 0u && (reinterpret_cast<uintptr_t>(ep.logits) & 15u) == 0u;
    float v[4];
    if (vec) {
        const float4 t = (id < ep.V) ? *reinterpret_cast<const float4*>(lrow + id)
                                     : make_float4(-INFINITY, -INFINITY, -INFINITY, -INFINITY);
        v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
    } else {
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) v[i] = (id + i < ep.V) ? lrow[id + i] : -INFINITY;
    }
    // the row this workgroup copies, if there is one
    const uint32_t crow = blockIdx.y * ((ep.ntile + kEpiTiles - 1u) / kEpiTiles) + blockIdx.x;
    const bool copies = rc.dst && crow < rc.n && threadIdx.x < kRowWords;
    uint32_t row_word = 0u;
    if (copies) row_word = reinterpret_cast<const uint32_t*>(rc.src ? rc.src + crow : &rc.inl[crow])[threadIdx.x];
    bool changed = false;
    // the four ids share one word of the bit masks
    if (mods && id < ep.V) {
        const DevRow& row = ep.rows[b];
        uint32_t cnt[4] = {0u, 0u, 0u, 0u}, has_bias[4] = {0u, 0u, 0u, 0u};
        float bias[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if ((row.has_mods & 1u) && ep.hcount) {
            uint32_t* wp = ep.hbits + (size_t)b * ep.hbw + (id >> 5);
            const uint32_t hw = *wp;
            if ((id & 31u) == 0u && hw != 0u) *wp = 0u;  // read by this wave's lanes only
            const uint32_t nib = (hw >> (id & 31u)) & 15u;
            if (nib) {
                uint32_t* cp = ep.hcount + (size_t)b * ep.V + id;
#pragma unroll
                for (uint32_t i = 0; i < 4; ++i) cnt[i] = ((nib >> i) & 1u) ? cp[i] : 0u;
#pragma unroll
                for (uint32_t i = 0; i < 4; ++i)
                    if (cnt[i]) cp[i] = 0u;  // zero again for the next step
            }
        }
        if ((row.has_mods & 2u) && ep.block_start) {
            const uint32_t* bs = ep.block_start + (size_t)b * (ep.ntile + 1u) + tile;
            const ModEntry* me = ep.mods + (size_t)b * ep.mod_cap;
            for (uint32_t k = bs[0], e = bs[1]; k < e; ++k) {
                const ModEntry t = me[k];
#pragma unroll
                for (uint32_t i = 0; i < 4; ++i)
                    if (t.id == id + i) { bias[i] = t.bias; has_bias[i] = 1u; }
            }
        }
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i)
            if (cnt[i] || has_bias[i]) {
                const float n = apply_entry(v[i], ModEntry{id + i, cnt[i], bias[i], has_bias[i]}, row, ep.rep_limit);
                changed = changed || __float_as_uint(n) != __float_as_uint(v[i]);
                v[i] = n;
            }
    }
    if (ep.ban && id < ep.V) {
        const uint32_t nib = (ep.ban[(size_t)b * ep.ban_stride + (id >> 5)] >> (id & 31u)) & 15u;
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i)
            if ((nib >> i) & 1u) {
                changed = changed || v[i] != -INFINITY;
                v[i] = -INFINITY;
            }
    }
    if (!vec) {  // ids past the vocabulary (a ban bit may be set there)
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i)
            if (id + i >= ep.V) v[i] = -INFINITY;
    }
    if (changed) {
        if (vec) {
            *reinterpret_cast<float4*>(lrow + id) = make_float4(v[0], v[1], v[2], v[3]);
        } else {
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i)
                if (id + i < ep.V) lrow[id + i] = v[i];
        }
    }
    const auto fmx = [](float a, float c) { return fmaxf(a, c); };
    const float m = row16_reduce(fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3])), fmx);
    uint32_t arg = 0xFFFFFFFFu;
#pragma unroll
    for (int i = 3; i >= 0; --i) arg = (v[i] == m) ? id + (uint32_t)i : arg;
    arg = row16_reduce(arg, [](uint32_t a, uint32_t c) { return min(a, c); });
    float sm = -INFINITY, mn = INFINITY, se = 0.0f;
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
        sm = fmaxf(sm, id + i == arg ? -INFINITY : v[i]);  // a repeat of the maximum counts
        mn = fminf(mn, v[i] == -INFINITY ? INFINITY : v[i]);
    }
    sm = row16_reduce(sm, fmx);
    mn = row16_reduce(mn, [](float a, float c) { return fminf(a, c); });
    if (!ep.no_sumexp) {
        if (m != -INFINITY) {
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) se += __expf(v[i] - m);
        }
        se = row16_reduce(se, [](float a, float c) { return a + c; });
    }
    if ((lane & 15u) == 0u && tile < ep.ntile) {
        BlockPartial bp;
        bp.max = m;
        bp.arg = arg;
        bp.sumexp = se;
        bp.minf = mn;
        bp.smax = sm;
        ep.partials[(size_t)b * ep.ntile + tile] = bp;
    }
    if (copies) reinterpret_cast<uint32_t*>(rc.dst + crow)[threadIdx.x] = row_word;
}

void launch_logits_epilogue(const Head& h, int batch, const EpiArgs& ep, const RowCopy& rc, bool mods, hipStream_t st) {
    hipLaunchKernelGGL(k_logits_epilogue, dim3((h.ntile + kEpiTiles - 1u) / kEpiTiles, (unsigned)batch), dim3(64 * kEpiWaves), 0, st,
                       ep, rc, mods ? 1u : 0u);
    check_hip(hipGetLastError(), "logits epilogue");
}

}  // namespace tdt
