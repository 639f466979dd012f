// moe_prefill.hip -- prefill MoE block over T token rows on gfx950.
//
// The reference runs prefill layer-major in chunks of 64 tokens
// (prefill.cpp:308-453): per token RMSNorm + router + top-k (:319-332), the
// per-expert token lists built by union_add (:38-68), one batched FFN per
// touched expert (metal_bridge.mm:544-645) and a weighted scatter into
// routed_out (:380-385) that is added to hidden (:446-451).  Here the whole
// batch of tokens is one pass (tokens are independent, so the grouping only
// changes fp32 summation order):
//
//   k_route        RMSNorm + fp32 router + exact top-k for TB tokens per
//                  block; writes the normed rows as the GEMM's f16 planes
//                  (the split below) and ids/weights.
//   k_split_rows   per row: power-of-two scale 2^e with |x| < 2^e and the
//                  f16 hi/lo planes of x * 2^-e (hi + lo carries 22 bits),
//                  columns of every 8 in the order 0 2 4 6 1 3 5 7.
//   k_perm_count, k_perm_scatter  stable counting sort of the T*k (token,
//                  rank) pairs by expert, one workgroup per segment of pairs,
//                  and the GEMMs' work lists (k_permute: one workgroup, with the
//                  union order by first appearance, for callers that ask for
//                  the permute's outputs and for batches of a few segments).
//   k_grouped_reg  per unit of up to 64 pairs of an expert: [pairs x K] x [K x
//                  rows] tiles (128 gate + 128 up rows, or 256 down rows, per
//                  block) on MFMA v_mfma_f32_16x16x32_f16, weights streamed into
//                  registers, activation rows through LDS (k_grouped_mm, with
//                  the weights through LDS too, where a row has an odd number
//                  of groups or the grid is small).  Weights enter exactly as
//                  (2c - 15)/8 (f16), activations as hi and lo planes (two
//                  MFMAs into one fp32 accumulator); each 64-column group adds
//                  s_g * sum, the row scale 8 * 2^e / 15 closes the dot
//                  (kernels.metal:90-105, 140-145).  Gate+up runs with SiLU
//                  and writes h per (token, rank) pair; down writes y per pair.
//   k_combine_pairs hidden[t] += sum_r w[t][r] * y[t*k + r] in rank order.
//
// Blocks of one expert are mapped to one XCD (block id mod 8), so its token
// rows stay in that XCD's L2 and its weights are shared there by its passes.
#include <algorithm>
#include <type_traits>

#include "device_common.hpp"
#include "kernels.hpp"
#include "topk.hpp"

namespace smoe {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

// ---------------------------------------------------------------------------
// 8 consecutive columns x[0..7] of a row with |x| < 2^e -> f16 planes hi, lo of
// x * 2^-e (hi + lo carries 22 bits), in the column order 0 2 4 6 1 3 5 7 in
// which q4_codes_to_f16 unpacks a word of codes.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void split8_f16(const float* x, int e, uint4& hi, uint4& lo)
{
    const float xs[8] = {x[0], x[2], x[4], x[6], x[1], x[3], x[5], x[7]};
    uint32_t h2[4], l2[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t hb[2], lb[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const float xv = __builtin_ldexpf(xs[2 * i + u], -e);
            const _Float16 h = static_cast<_Float16>(xv);
            hb[u] = __builtin_bit_cast(uint16_t, h);
            lb[u] = __builtin_bit_cast(uint16_t, static_cast<_Float16>(xv - static_cast<float>(h)));
        }
        h2[i] = hb[0] | (hb[1] << 16);
        l2[i] = lb[0] | (lb[1] << 16);
    }
    hi = make_uint4(h2[0], h2[1], h2[2], h2[3]);
    lo = make_uint4(l2[0], l2[1], l2[2], l2[3]);
}

// ---------------------------------------------------------------------------
// k_route: RMSNorm (common.hpp:245-256) + router (common.hpp:293-306) +
// softmax/top-k (scout.cpp:77-123) for TB tokens per block of ROUTE_WAVES
// waves.  Every wave normalises all TB tokens (lane l owns the 32-column
// chunks l + 64 j) and computes router rows w, w + ROUTE_WAVES, ... for all of
// them; wave t then selects the experts of token t, and (in the group's
// first block) writes token t's normed row as the GEMM's f16 planes.  With
// ES > 1 (short batches) the E router rows of a token group are split over
// ES blocks, so each wave has few rows and all their loads in flight at once:
// the blocks write their logits with agent-scope stores, wait for them, and
// add themselves to a device-scope counter per token group; the block that
// finds the count at ES - 1 modulo ES runs the group's top-k on agent-scope
// loads of the logits (no device-wide fence anywhere).  Where the registers
// allow (HAND below), wave t alone reads and normalises token t and hands it
// to the other waves through LDS, and every wave requests its first router
// rows before that, so the hidden rows' and the router rows' round trips
// overlap (same bits; 64 tokens of the 235B shape 16.1 -> 13.3 us, 512 of the
// 30B shape 20.3 -> 18.1 us).
// ---------------------------------------------------------------------------
constexpr int ROUTE_WAVES = 8;

template <int CPL, int TB, int VPL, int ES>
__global__ __launch_bounds__(ROUTE_WAVES * WAVE)
void k_route(MoeDims d, LayerDesc L, const float* __restrict__ hidden, uint32_t T, uint16_t* __restrict__ x_hi,
             uint16_t* __restrict__ x_lo, float* __restrict__ x_sc, uint32_t* __restrict__ ids,
             float* __restrict__ w, float* __restrict__ logits, uint32_t* __restrict__ counters)
{
    // router rows per reduction batch (RPB * TB values); with ES > 1 a wave
    // has at most 4 rows (E <= 128 at ES = 4)
    constexpr int RPB = ES > 1 ? 4 : 16 / TB;
    // the counters advance by ES per launch and token group, and one array
    // serves every launch: a single split factor keeps their residues aligned
    static_assert(ES == 1 || ES == 4, "one split factor for the route counters");
    __shared__ float s_logit[TB][SMOE_TOPK_MAX_N];
    __shared__ uint2 s_slots[TB][TOPK_SLOTS];
    __shared__ uint32_t s_last;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const uint32_t g = blockIdx.x / ES, eg = blockIdx.x % ES;
    const uint32_t t0 = g * TB;
    const uint32_t rows_per = (d.E + ES - 1) / ES, rbeg = eg * rows_per, rend = min(d.E, rbeg + rows_per);
    const uint32_t D = d.D, nch = D >> 5;

    // router rows per load group (see below)
    constexpr int RG_FIT = (208 - 32 * TB * CPL) / (16 * CPL);
    constexpr int RG_ALL = RG_FIT >= RPB ? RPB : RG_FIT >= 8 ? 8 : RG_FIT >= 4 ? 4 : RG_FIT >= 2 ? 2 : 1;
    // HAND: waves 0 .. TB - 1 normalise the tokens and hand them over through
    // LDS while every wave requests its first group of router rows (where that
    // fits the registers without spills: one chunk a lane, or one token at two;
    // E <= 128)
    constexpr bool HAND = ES > 1 || (VPL == 2 && (CPL == 1 || (CPL == 2 && TB == 1)));
    // (two rows a group where a wave's hidden chunks are live beside them)
    constexpr int RG = HAND && CPL > 1 && RG_ALL > 2 ? 2 : RG_ALL;
    static_assert(RPB % RG == 0, "row groups of a batch");
    const uint32_t rfirst = rbeg + wv * RPB;
    uint4 rws[RG][CPL][4];
    float a[TB][CPL][32];
    if constexpr (HAND) {
        // wave t < TB normalises token t (and, in the token group's first
        // block, writes its f16 planes) and hands it to the other waves
        // through LDS; every wave requests its router rows before that, so the
        // round trips overlap and each token is normalised once, not by every wave
        __shared__ __align__(16) float4 s_a[TB][CPL][8][WAVE];
        float4 x[CPL][8];
        uint4 gw[CPL][4];
        if (wv < TB) {
            const float* hv = hidden + static_cast<size_t>(min(t0 + wv, T - 1)) * D;
#pragma unroll
            for (int j = 0; j < CPL; ++j) {
                const uint32_t c = min(lane + WAVE * j, nch - 1);
#pragma unroll
                for (int q = 0; q < 8; ++q) x[j][q] = load_f4(hv + c * 32 + q * 4);
#pragma unroll
                for (int q = 0; q < 4; ++q) gw[j][q] = load_u4(L.norm_w + c * 32 + q * 8);
            }
        }
        if (rfirst < rend) {
#pragma unroll
            for (int ii = 0; ii < RG; ++ii) {
                const uint16_t* wr = L.router_w + static_cast<size_t>(min(rfirst + ii, rend - 1)) * D;
#pragma unroll
                for (int j = 0; j < CPL; ++j) {
                    const uint32_t c = min(lane + WAVE * j, nch - 1);
#pragma unroll
                    for (int q = 0; q < 4; ++q) rws[ii][j][q] = load_u4(wr + c * 32 + q * 8);
                }
            }
        }
        if (wv < TB) {
            float ss = 0.f;
#pragma unroll
            for (int j = 0; j < CPL; ++j) {
                const bool ok = lane + WAVE * j < nch;
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    if (!ok) x[j][q] = make_float4(0.f, 0.f, 0.f, 0.f);
                    ss = fmaf(x[j][q].x, x[j][q].x, ss);
                    ss = fmaf(x[j][q].y, x[j][q].y, ss);
                    ss = fmaf(x[j][q].z, x[j][q].z, ss);
                    ss = fmaf(x[j][q].w, x[j][q].w, ss);
                }
            }
            ss = wave_sum(ss);
            const float inv = 1.0f / sqrtf(ss / static_cast<float>(D) + 1e-6f);
#pragma unroll
            for (int j = 0; j < CPL; ++j) {
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    const uint32_t g0 = (q & 1) ? gw[j][q >> 1].z : gw[j][q >> 1].x;
                    const uint32_t g1 = (q & 1) ? gw[j][q >> 1].w : gw[j][q >> 1].y;
                    a[0][j][4 * q + 0] = (x[j][q].x * inv) * bf16_to_f32(g0 & 0xFFFFu);
                    a[0][j][4 * q + 1] = (x[j][q].y * inv) * bf16_to_f32(g0 >> 16);
                    a[0][j][4 * q + 2] = (x[j][q].z * inv) * bf16_to_f32(g1 & 0xFFFFu);
                    a[0][j][4 * q + 3] = (x[j][q].w * inv) * bf16_to_f32(g1 >> 16);
                }
#pragma unroll
                for (int q = 0; q < 8; ++q)
                    s_a[wv][j][q][lane] = make_float4(a[0][j][4 * q], a[0][j][4 * q + 1], a[0][j][4 * q + 2],
                                                      a[0][j][4 * q + 3]);
            }
            if (eg == 0 && t0 + wv < T) {
                float amax = 0.f;
#pragma unroll
                for (int j = 0; j < CPL; ++j)
                    if (lane + WAVE * j < nch) {
#pragma unroll
                        for (int k = 0; k < 32; ++k) amax = fmaxf(amax, fabsf(a[0][j][k]));
                    }
                amax = wave_max(amax);
                const int e = amax > 0.f ? __builtin_amdgcn_frexp_expf(amax) : 0;
                const size_t row = static_cast<size_t>(t0 + wv) * D;
#pragma unroll
                for (int j = 0; j < CPL; ++j) {
                    if (lane + WAVE * j >= nch) continue;
#pragma unroll
                    for (int b = 0; b < 4; ++b) {
                        const size_t o = row + (lane + WAVE * j) * 32 + 8 * b;
                        uint4 hv4, lv4;
                        split8_f16(&a[0][j][8 * b], e, hv4, lv4);
                        *reinterpret_cast<uint4*>(x_hi + o) = hv4;
                        *reinterpret_cast<uint4*>(x_lo + o) = lv4;
                    }
                }
                if (lane == 0) x_sc[t0 + wv] = __builtin_ldexpf(1.0f, e);
            }
        }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < TB; ++t)
#pragma unroll
            for (int j = 0; j < CPL; ++j)
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    const float4 v = s_a[t][j][q][lane];
                    a[t][j][4 * q] = v.x;
                    a[t][j][4 * q + 1] = v.y;
                    a[t][j][4 * q + 2] = v.z;
                    a[t][j][4 * q + 3] = v.w;
                }
    } else
#pragma unroll
    for (int t = 0; t < TB; ++t) {
        const float* hv = hidden + static_cast<size_t>(min(t0 + t, T - 1)) * D;

        float4 x[CPL][8];
        uint4 g[CPL][4];
#pragma unroll
        for (int j = 0; j < CPL; ++j) {
            const uint32_t c = min(lane + WAVE * j, nch - 1);
#pragma unroll
            for (int q = 0; q < 8; ++q) x[j][q] = load_f4(hv + c * 32 + q * 4);
#pragma unroll
            for (int q = 0; q < 4; ++q) g[j][q] = load_u4(L.norm_w + c * 32 + q * 8);
        }
        float ss = 0.f;
#pragma unroll
        for (int j = 0; j < CPL; ++j) {
            const bool ok = lane + WAVE * j < nch;
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                if (!ok) x[j][q] = make_float4(0.f, 0.f, 0.f, 0.f);
                ss = fmaf(x[j][q].x, x[j][q].x, ss);
                ss = fmaf(x[j][q].y, x[j][q].y, ss);
                ss = fmaf(x[j][q].z, x[j][q].z, ss);
                ss = fmaf(x[j][q].w, x[j][q].w, ss);
            }
        }
        ss = wave_sum(ss);
        const float inv = 1.0f / sqrtf(ss / static_cast<float>(D) + 1e-6f);
#pragma unroll
        for (int j = 0; j < CPL; ++j) {
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const uint32_t g0 = (q & 1) ? g[j][q >> 1].z : g[j][q >> 1].x;
                const uint32_t g1 = (q & 1) ? g[j][q >> 1].w : g[j][q >> 1].y;
                a[t][j][4 * q + 0] = (x[j][q].x * inv) * bf16_to_f32(g0 & 0xFFFFu);
                a[t][j][4 * q + 1] = (x[j][q].y * inv) * bf16_to_f32(g0 >> 16);
                a[t][j][4 * q + 2] = (x[j][q].z * inv) * bf16_to_f32(g1 & 0xFFFFu);
                a[t][j][4 * q + 3] = (x[j][q].w * inv) * bf16_to_f32(g1 >> 16);
            }
        }
        // wave t of the group's first block writes token t's normed row as the
        // grouped GEMM's f16 planes (the split of k_split_rows, same values)
        if (wv == t && eg == 0 && t0 + t < T) {
            float amax = 0.f;
#pragma unroll
            for (int j = 0; j < CPL; ++j)
                if (lane + WAVE * j < nch) {
#pragma unroll
                    for (int k = 0; k < 32; ++k) amax = fmaxf(amax, fabsf(a[t][j][k]));
                }
            amax = wave_max(amax);
            const int e = amax > 0.f ? __builtin_amdgcn_frexp_expf(amax) : 0;
            const size_t row = static_cast<size_t>(t0 + t) * D;
#pragma unroll
            for (int j = 0; j < CPL; ++j) {
                if (lane + WAVE * j >= nch) continue;
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    const size_t o = row + (lane + WAVE * j) * 32 + 8 * b;
                    uint4 hv, lv;
                    split8_f16(&a[t][j][8 * b], e, hv, lv);
                    *reinterpret_cast<uint4*>(x_hi + o) = hv;
                    *reinterpret_cast<uint4*>(x_lo + o) = lv;
                }
            }
            if (lane == 0) x_sc[t0 + t] = __builtin_ldexpf(1.0f, e);
        }
    }
    // router rows of this wave, RPB at a time; lane l ends up with value
    // l >> VSH of the batch (value v = row_i * TB + t)
    // The rows are requested RG at a time before any of them is used, so their
    // loads are in flight together (row by row, the compiler waited out one L2
    // round trip per row: 21.4 us for the route at 512 tokens of the 30B
    // shape).  RG: as many rows as fit beside the normed activations
    // (TB * CPL * 32 values) in about 208 VGPRs, 16 CPL registers a row.
    // With ES > 1 the first group was requested before the norm (above).
    for (uint32_t r0 = rfirst; r0 < rend; r0 += ROUTE_WAVES * RPB) {
        float part[RPB * TB];
#pragma unroll
        for (int i = 0; i < RPB; ++i) {
            if (i % RG == 0 && (!HAND || i > 0 || r0 != rfirst)) {
#pragma unroll
                for (int ii = 0; ii < RG; ++ii) {
                    const uint16_t* wr = L.router_w + static_cast<size_t>(min(r0 + i + ii, rend - 1)) * D;
#pragma unroll
                    for (int j = 0; j < CPL; ++j) {
                        const uint32_t c = min(lane + WAVE * j, nch - 1);
#pragma unroll
                        for (int q = 0; q < 4; ++q) rws[ii][j][q] = load_u4(wr + c * 32 + q * 8);
                    }
                }
            }
            const uint4 (&rw)[CPL][4] = rws[i % RG];
#pragma unroll
            for (int t = 0; t < TB; ++t) {
                float acc = 0.f;
#pragma unroll
                for (int j = 0; j < CPL; ++j) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const uint32_t w4[4] = {rw[j][q].x, rw[j][q].y, rw[j][q].z, rw[j][q].w};
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            acc = fmaf(bf16_to_f32(w4[u] & 0xFFFFu), a[t][j][8 * q + 2 * u], acc);
                            acc = fmaf(bf16_to_f32(w4[u] >> 16), a[t][j][8 * q + 2 * u + 1], acc);
                        }
                    }
                }
                part[i * TB + t] = acc;
            }
        }
        const float tot = wave_sum_rows<RPB * TB>(part);
        constexpr int VSH = 6 - ilog2(RPB * TB);   // lane l holds the total of value l >> VSH
        const uint32_t v = lane >> VSH;
        const uint32_t row = r0 + v / TB;
        if ((lane & ((1 << VSH) - 1)) == 0 && row < rend && row < r0 + RPB) {
            if (ES == 1) s_logit[v % TB][row] = tot;
            else if (t0 + v % TB < T)   // written through to the agent's coherence point
                __hip_atomic_store(&logits[static_cast<size_t>(t0 + v % TB) * d.E + row], tot, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    if (ES > 1) {
        // every wave's agent-scope stores complete before the block counts
        // itself (no device-wide fence: that writes back and invalidates the
        // whole L2 of the XCD)
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
        asm volatile("" ::: "memory");
        __syncthreads();
        // the count is kept modulo ES (ES divides 2^32): no reset between launches
        if (threadIdx.x == 0) s_last = atomicAdd(&counters[g], 1u) % ES == ES - 1;
        __syncthreads();
        if (!s_last) return;
    } else {
        __syncthreads();
    }
    if (wv < TB && t0 + wv < T) {
        float p[VPL];
#pragma unroll
        for (int j = 0; j < VPL; ++j) {
            const uint32_t pos = lane + WAVE * j;
            p[j] = pos >= d.E ? -INFINITY
                   : ES == 1  ? s_logit[wv][pos]
                              : __hip_atomic_load(&logits[static_cast<size_t>(t0 + wv) * d.E + pos],
                                                  __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        uint32_t my_id;
        float my_w;
        const uint32_t count = topk_latency<VPL>(p, d.E, d.K, d.norm_topk, my_id, my_w, s_slots[wv]);
        if (static_cast<uint32_t>(lane) < count) {
            ids[static_cast<size_t>(t0 + wv) * d.K + lane] = my_id;
            w[static_cast<size_t>(t0 + wv) * d.K + lane] = my_w;
        }
    }
}

// ---------------------------------------------------------------------------
// k_split_rows: src [rows x cols] fp32 -> f16 planes hi/lo of x * 2^-e with
// |x| < 2^e over the row, and scale[row] = 2^e.  hi + lo carries 22 bits of
// x * 2^-e (f16 subnormals below 2^-14 still hold x to 2^-25 of the row max).
// Within every 8 columns the planes hold the columns in the order
// 0 2 4 6 1 3 5 7, the order in which q4_codes_to_f16 unpacks a word of
// codes (the even codes, then the odd ones).  One wave per row, 8 columns
// per lane; rows of 1025 to 2048 columns are read once (kept in registers
// between the maximum and the split).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256)
void k_split_rows(const float* __restrict__ src, uint32_t rows, uint32_t cols, uint16_t* __restrict__ hi,
                  uint16_t* __restrict__ lo, float* __restrict__ scale)
{
    const int lane = threadIdx.x & 63;
    for (uint32_t r = blockIdx.x * 4 + (threadIdx.x >> 6); r < rows; r += gridDim.x * 4) {
        const float* x = src + static_cast<size_t>(r) * cols;
        float amax = 0.f;
        if (cols > 2 * WAVE * 8 && cols <= 4 * WAVE * 8) {
            // the row's 8-column pieces of this lane stay in registers: one read of the row
            // (at 1536 columns 4.5 against 5.9 us for 512 rows; at 768 the second read is
            // cheaper than the half-line loads of this mapping, 5.8 against 6.1 us)
            float4 v[4][2];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t c = lane * 8 + WAVE * 8 * i;
                if (c < cols) {
                    v[i][0] = load_f4(x + c);
                    v[i][1] = load_f4(x + c + 4);
                    const float4 a = v[i][0], b = v[i][1];
                    amax = fmaxf(amax, fmaxf(fmaxf(fmaxf(fabsf(a.x), fabsf(a.y)), fmaxf(fabsf(a.z), fabsf(a.w))),
                                             fmaxf(fmaxf(fabsf(b.x), fabsf(b.y)), fmaxf(fabsf(b.z), fabsf(b.w)))));
                }
            }
            amax = wave_max(amax);
            const int e = amax > 0.f ? __builtin_amdgcn_frexp_expf(amax) : 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t c = lane * 8 + WAVE * 8 * i;
                if (c < cols) {
                    const float xv[8] = {v[i][0].x, v[i][0].y, v[i][0].z, v[i][0].w,
                                         v[i][1].x, v[i][1].y, v[i][1].z, v[i][1].w};
                    uint4 hv, lv;
                    split8_f16(xv, e, hv, lv);
                    const size_t o = static_cast<size_t>(r) * cols + c;
                    *reinterpret_cast<uint4*>(hi + o) = hv;
                    *reinterpret_cast<uint4*>(lo + o) = lv;
                }
            }
            if (lane == 0) scale[r] = __builtin_ldexpf(1.0f, e);
            continue;
        }
        for (uint32_t c = lane * 4; c < cols; c += WAVE * 4) {
            const float4 v = load_f4(x + c);
            amax = fmaxf(amax, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
        }
        amax = wave_max(amax);
        const int e = amax > 0.f ? __builtin_amdgcn_frexp_expf(amax) : 0;
        for (uint32_t c = lane * 8; c < cols; c += WAVE * 8) {
            const float4 v0 = load_f4(x + c), v1 = load_f4(x + c + 4);
            const float xv[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
            uint4 hv, lv;
            split8_f16(xv, e, hv, lv);
            const size_t o = static_cast<size_t>(r) * cols + c;
            *reinterpret_cast<uint4*>(hi + o) = hv;
            *reinterpret_cast<uint4*>(lo + o) = lv;
        }
        if (lane == 0) scale[r] = __builtin_ldexpf(1.0f, e);
    }
}

// ---------------------------------------------------------------------------
// k_permute: stable counting sort of the P = T*k pairs p = t*k + r by expert
// ids[p] (prefill.cpp:38-68 builds the same per-expert lists, ascending token
// order), in one workgroup.  Chunk c = pairs [64c, 64c + 64) is one wave's
// step: per-(expert, chunk) counts in LDS, prefix over (expert, chunk), then
// each pair's slot = prefix + its rank among equal ids earlier in the chunk.
// The count table is [expert][chunk] with an odd row stride, so the threads
// that scan one expert's chunks read different banks (the [chunk][expert]
// table put them all in one: 14.2 -> 11.6 us at 512 tokens of the 30B shape).
// Union order (first appearance, token-major, prefill.cpp:55-68) ranks the
// touched experts by their first pair.  ids >= E are skipped and flagged in
// err (bit 1).  lists (optional) receives the grouped GEMMs' work lists.
// ---------------------------------------------------------------------------
constexpr int PERM_THREADS = 1024;

// The grouped GEMMs' work lists: units of up to cap (unit_cap) pairs of one
// expert, an expert's M pairs in as few units as cap allows, of equal numbers of
// 16-row tiles.  First the units of more than 16 rows, then those of 16, experts
// ascending in either: what is left for the end of a launch is short (in the
// order of the experts alone 32 Zipf-routed tokens of the 30B shape took 89 us
// against 81, 200 of them 141 against 117, 150 tokens of 60 experts 80 against
// 73).  An XCD takes consecutive long units and consecutive short ones (unit_share;
// block id mod 8 is a block's XCD), so an expert's blocks run together on one XCD
// and share its activation rows and, between its units, its weights in the L2.
// The record of the j-th unit of XCD x stands at 8 j + x, all 8 slots of every j
// the grid covers are written (no pairs: no unit), and a record holds all that a
// block needs: one scalar load, then the pairs and the weights.
//
// The tables over the experts hold two counts a word: long units before the
// expert's in the low half, short ones (after all the long ones) in the high half.
__device__ __forceinline__ uint32_t unit_count(uint32_t M, uint32_t cap) { return (M + cap - 1u) / cap; }
__device__ __forceinline__ uint32_t unit_rows(uint32_t M, uint32_t cap)
{
    const uint32_t tiles = (M + 15u) >> 4, n = unit_count(M, cap);
    return n ? 16u * ((tiles + n - 1u) / n) : 16u;
}
__device__ __forceinline__ uint32_t unit_pair(uint32_t M, uint32_t cap)
{
    return unit_count(M, cap) << (M > 16u ? 0u : 16u);
}

// One wave, EPL experts a lane: exclusive scans of the E experts' totals s_tot into
// s_off [E + 1] (pairs) and s_unit [2][E + 1] (units of up to 64, of up to 32
// pairs), and the caps of the two work lists.
template <int EPL>
__device__ __forceinline__ void scan_units_n(const uint32_t* s_tot, uint32_t E, const UnitLists& lists, uint32_t* s_off,
                                             uint32_t* s_unit, uint32_t* s_cap)
{
    const uint32_t lane = threadIdx.x & 63;
    uint32_t tot[EPL], u64 = 0, u32 = 0, sum = 0;
#pragma unroll
    for (int i = 0; i < EPL; ++i) {
        const uint32_t e = EPL * lane + i;
        tot[i] = e < E ? s_tot[e] : 0u;
        sum += tot[i];
        u64 += unit_pair(tot[i], 64u);
        u32 += unit_pair(tot[i], 32u);
    }
    auto inclusive = [&](uint32_t v) {
        for (uint32_t dlt = 1; dlt < WAVE; dlt <<= 1) {
            const uint32_t o = __shfl_up(v, dlt);
            if (lane >= dlt) v += o;
        }
        return v;
    };
    const uint32_t i_tot = inclusive(sum), i64 = inclusive(u64), i32 = inclusive(u32);
    const uint32_t n64 = readlane_u32(i64, WAVE - 1), n32 = readlane_u32(i32, WAVE - 1);
    const uint32_t P = readlane_u32(i_tot, WAVE - 1);
    // (the short units' counts start after all the long ones)
    uint32_t run = i_tot - sum, run64 = i64 - u64 + (n64 << 16), run32 = i32 - u32 + (n32 << 16);
#pragma unroll
    for (int i = 0; i < EPL; ++i) {
        const uint32_t e = EPL * lane + i;
        if (e < E) {
            s_off[e] = run;
            s_unit[e] = run64;
            s_unit[E + 1 + e] = run32;
        }
        run += tot[i];
        run64 += unit_pair(tot[i], 64u);
        run32 += unit_pair(tot[i], 32u);
    }
    if (lane == WAVE - 1) {
        s_off[E] = run;
        s_unit[E] = run64;
        s_unit[2 * E + 1] = run32;
    }
    if (lane < 2)
        s_cap[lane] = unit_cap(P, (n64 & 0xFFFFu) + (n64 >> 16), (n32 & 0xFFFFu) + (n32 >> 16),
                               lane == 0 ? lists.tiles[0] : lists.tiles[1]);
}
__device__ __forceinline__ void scan_units(const uint32_t* s_tot, uint32_t E, const UnitLists& lists, uint32_t* s_off,
                                           uint32_t* s_unit, uint32_t* s_cap)
{
    if (E <= 64) scan_units_n<1>(s_tot, E, lists, s_off, s_unit, s_cap);
    else if (E <= 128) scan_units_n<2>(s_tot, E, lists, s_off, s_unit, s_cap);
    else scan_units_n<8>(s_tot, E, lists, s_off, s_unit, s_cap);
}

// a workgroup writes the records of both lists (s_off, s_unit, s_cap: scan_units):
// x = expert | rows of a pass << 16, y = first pair, z = pairs
__device__ __forceinline__ void write_units(const uint32_t* s_off, const uint32_t* s_unit, uint32_t E,
                                            const uint32_t* s_cap, const UnitLists& lists)
{
    for (uint32_t k = threadIdx.x; k < lists.slots[0] + lists.slots[1]; k += blockDim.x) {
        const bool down = k >= lists.slots[0];
        const uint32_t i = down ? k - lists.slots[0] : k, cap = s_cap[down ? 1 : 0];
        const uint32_t* tab = s_unit + (cap == 32u ? E + 1u : 0u);
        const uint32_t n_long = tab[E] & 0xFFFFu, n_short = (tab[E] >> 16) - n_long;
        const uint32_t j = i >> 3;
        const UnitShare xcd = unit_share(i & 7u, n_long, n_short);
        uint4 rec = make_uint4(0u, 0u, 0u, 0u);
        if (j < xcd.nl + xcd.ns) {
            const uint32_t sh = j < xcd.nl ? 0u : 16u, u = j < xcd.nl ? xcd.l0 + j : n_long + xcd.s0 + (j - xcd.nl);
            auto first = [&](uint32_t e) { return (tab[e] >> sh) & 0xFFFFu; };
            uint32_t e = 0, hi = E;              // the expert: first(e) <= u < first(e + 1)
            while (hi - e > 1) {
                const uint32_t mid = (e + hi) >> 1;
                if (first(mid) <= u) e = mid;
                else hi = mid;
            }
            const uint32_t M = s_off[e + 1] - s_off[e], rows = unit_rows(M, cap), m0 = (u - first(e)) * rows;
            rec = make_uint4(e | (rows << 16), s_off[e] + m0, min(M - m0, rows), 0u);
        }
        lists.units[k] = rec;
    }
}

__global__ __launch_bounds__(PERM_THREADS)
void k_permute(const uint32_t* __restrict__ ids, const float* __restrict__ w, uint32_t P, uint32_t K, uint32_t E,
               uint32_t* __restrict__ offsets, uint32_t* __restrict__ sorted_pairs,
               uint32_t* __restrict__ sorted_tokens, float* __restrict__ sorted_w, uint32_t* __restrict__ union_ids,
               uint32_t* __restrict__ union_size, UnitLists lists, uint32_t* __restrict__ err)
{
    extern __shared__ uint32_t s_mem[];
    __shared__ uint32_t s_cap[2];
    // the count table is [E][C | 1]: the odd row stride puts a chunk's experts,
    // and the chunks one expert's threads read, in different banks
    const uint32_t C = (P + 63) / 64, CS = C | 1u;
    uint32_t* s_cnt = s_mem;               // [E x CS]
    uint32_t* s_first = s_cnt + CS * E;    // [E]
    uint32_t* s_tot = s_first + E;         // [E]
    uint32_t* s_off = s_tot + E;           // [E + 1]
    uint32_t* s_unit = s_off + E + 1;      // [2][E + 1]
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    constexpr int NW = PERM_THREADS / WAVE;

    for (uint32_t i = threadIdx.x; i < CS * E; i += PERM_THREADS) s_cnt[i] = 0;
    for (uint32_t i = threadIdx.x; i < E; i += PERM_THREADS) s_first[i] = 0xFFFFFFFFu;
    // each wave takes chunks wv, wv + NW, ...; the ids of up to PERM_BATCH of
    // them are loaded together (one memory round trip), and kept for the
    // scatter when one batch covers all of the wave's chunks
    constexpr int PERM_BATCH = 8;
    const bool one_batch = C <= NW * PERM_BATCH;
    uint32_t eid[PERM_BATCH];
    auto load_ids = [&](uint32_t c_first) {
#pragma unroll
        for (int k = 0; k < PERM_BATCH; ++k) {
            const uint32_t p = (c_first + k * NW) * 64 + lane;
            eid[k] = p < P ? ids[p] : 0xFFFFFFFFu;
        }
    };
    __syncthreads();
    for (uint32_t cb = wv; cb < C; cb += NW * PERM_BATCH) {
        load_ids(cb);
#pragma unroll
        for (int k = 0; k < PERM_BATCH; ++k) {
            const uint32_t c = cb + k * NW, p = c * 64 + lane;
            if (c >= C || p >= P) continue;
            const uint32_t e = eid[k];
            if (e < E) {
                atomicAdd(&s_cnt[e * CS + c], 1u);
                if (union_ids) atomicMin(&s_first[e], p);
            } else {
                atomicOr(err, 2u);
            }
        }
    }
    __syncthreads();
    // per expert: counts -> exclusive prefix over chunks.  S threads (a power
    // of two, in one wave) share an expert's C chunks in segments: segment sums,
    // an exclusive scan over the segments, then each chunk's prefix.
    {
        uint32_t S = 64;
        while (S > 1 && E * S > PERM_THREADS) S >>= 1;
        const uint32_t e = threadIdx.x / S, sg = threadIdx.x % S;
        const uint32_t Lc = (C + S - 1) / S;
        const uint32_t c0 = min(sg * Lc, C), c1 = min(c0 + Lc, C);
        uint32_t seg = 0;
        if (e < E)
            for (uint32_t c = c0; c < c1; ++c) seg += s_cnt[e * CS + c];
        // inclusive scan over the S segments of this expert (lanes e*S .. e*S + S - 1)
        uint32_t inc = seg;
        for (uint32_t dlt = 1; dlt < S; dlt <<= 1) {
            const uint32_t o = __shfl_up(inc, dlt, S);
            if (sg >= dlt) inc += o;
        }
        if (e < E) {
            uint32_t run = inc - seg;
            for (uint32_t c = c0; c < c1; ++c) {
                const uint32_t t = s_cnt[e * CS + c];
                s_cnt[e * CS + c] = run;
                run += t;
            }
            if (sg == S - 1) s_tot[e] = inc;
        }
    }
    __syncthreads();
    // expert offsets and units
    if (wv == 0) scan_units(s_tot, E, lists, s_off, s_unit, s_cap);
    __syncthreads();
    for (uint32_t e = threadIdx.x; e <= E; e += PERM_THREADS) offsets[e] = s_off[e];
    // scatter: rank among equal ids of lower lanes of the same chunk; the
    // lanes holding this lane's id are found bit by bit (one ballot per bit
    // of an id below E)
    uint32_t nbits = 1;
    while ((1u << nbits) < E) ++nbits;
    for (uint32_t cb = wv; cb < C; cb += NW * PERM_BATCH) {
      if (!one_batch) load_ids(cb);
#pragma unroll
      for (int k = 0; k < PERM_BATCH; ++k) {
        const uint32_t c = cb + k * NW;
        if (c >= C) break;
        const uint32_t p = c * 64 + lane;
        const uint32_t e = eid[k];
        const bool ok = e < E;
        uint64_t same = __ballot(ok);
        for (uint32_t b = 0; b < nbits; ++b) {
            const bool bit = (e >> b) & 1u;
            const uint64_t set = __ballot(ok && bit);
            same &= bit ? set : ~set;
        }
        const uint32_t rank = __popcll(same & ((1ull << lane) - 1ull));
        if (ok) {
            const uint32_t dst = s_off[e] + s_cnt[e * CS + c] + rank;
            sorted_pairs[dst] = p;
            if (sorted_tokens) sorted_tokens[dst] = p / K;
            if (sorted_w) sorted_w[dst] = w[p];
        }
      }
    }
    // union order: touched experts ranked by first appearance
    if (union_ids) {
        for (uint32_t e = threadIdx.x; e < E; e += PERM_THREADS) {
            if (s_tot[e] == 0) continue;
            uint32_t r = 0;
            for (uint32_t e2 = 0; e2 < E; ++e2) r += (s_tot[e2] != 0 && s_first[e2] < s_first[e]);
            union_ids[r] = e;
        }
    }
    if (union_size && threadIdx.x == 0) {
        uint32_t n = 0;
        for (uint32_t e = 0; e < E; ++e) n += s_tot[e] != 0;
        *union_size = n;
    }
    if (lists.units) write_units(s_off, s_unit, E, s_cap, lists);
}

// ---------------------------------------------------------------------------
// The permute of long batches, in segments of PERM_SEG_CHUNKS(E) chunks of 64
// pairs, one workgroup each (k_permute's tables of a whole long batch do not
// fit one workgroup's LDS, and one CU would take the scatter alone):
//   k_perm_count    per segment and expert: the number of its pairs;
//   k_perm_scatter  every workgroup adds up the counts of the segments before
//                   its own and of all of them, scans the totals into the
//                   expert offsets, and places its segment's pairs as
//                   k_permute does.  Workgroup 0 also writes the grouped
//                   GEMMs' work lists.
// A batch of one segment needs no counts from elsewhere: k_perm_scatter counts
// it itself (ONE) and is the only launch (64 tokens of the 30B shape 115.9 ->
// 113.5 us a call).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(PERM_THREADS)
void k_perm_count(const uint32_t* __restrict__ ids, uint32_t P, uint32_t E, uint32_t* __restrict__ seg_cnt,
                  uint32_t* __restrict__ err)
{
    __shared__ uint32_t s_cnt[SMOE_TOPK_MAX_N];
    for (uint32_t e = threadIdx.x; e < E; e += PERM_THREADS) s_cnt[e] = 0;
    __syncthreads();
    const uint32_t len = 64u * perm_seg_chunks(E), p0 = blockIdx.x * len, p1 = min(P, p0 + len);
    for (uint32_t p = p0 + threadIdx.x; p < p1; p += PERM_THREADS) {
        const uint32_t e = ids[p];
        if (e < E) atomicAdd(&s_cnt[e], 1u);
        else atomicOr(err, 2u);
    }
    __syncthreads();
    for (uint32_t e = threadIdx.x; e < E; e += PERM_THREADS)
        seg_cnt[static_cast<size_t>(blockIdx.x) * E + e] = s_cnt[e];
}

template <bool ONE>
__global__ __launch_bounds__(PERM_THREADS)
void k_perm_scatter(const uint32_t* __restrict__ ids, uint32_t P, uint32_t E, const uint32_t* __restrict__ seg_cnt,
                    uint32_t* __restrict__ sorted_pairs, UnitLists lists, uint32_t* __restrict__ err)
{
    extern __shared__ uint32_t s_mem[];
    __shared__ uint32_t s_cap[2];
    const uint32_t CH = perm_seg_chunks(E), CS = CH | 1u;
    uint32_t* s_cnt = s_mem;               // [E x CS]
    uint32_t* s_base = s_cnt + E * CS;     // [E] pairs of the expert in earlier segments
    uint32_t* s_tot = s_base + E;          // [E]
    uint32_t* s_off = s_tot + E;           // [E + 1]
    uint32_t* s_unit = s_off + E + 1;      // [2][E + 1]
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    constexpr uint32_t NW = PERM_THREADS / WAVE;
    const uint32_t seg = blockIdx.x, nseg = gridDim.x;
    for (uint32_t i = threadIdx.x; i < E * CS; i += PERM_THREADS) s_cnt[i] = 0;
    uint32_t eid[2];                       // this wave's chunks wv and wv + NW of the segment
#pragma unroll
    for (uint32_t k = 0; k < 2; ++k) {
        const uint32_t c = wv + k * NW, p = (seg * CH + c) * 64 + lane;
        eid[k] = c < CH && p < P ? ids[p] : 0xFFFFFFFFu;
    }
    for (uint32_t e = threadIdx.x; e < E; e += PERM_THREADS) {
        uint32_t before = 0, tot = 0;
        if constexpr (!ONE) {
#pragma unroll 8
            for (uint32_t s = 0; s < nseg; ++s) {
                const uint32_t n = seg_cnt[static_cast<size_t>(s) * E + e];
                tot += n;
                before += s < seg ? n : 0u;
            }
        }
        s_base[e] = before;
        s_tot[e] = tot;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < 2; ++k) {
        const uint32_t c = wv + k * NW;
        if (eid[k] < E) {
            atomicAdd(&s_cnt[eid[k] * CS + c], 1u);
            if constexpr (ONE) atomicAdd(&s_tot[eid[k]], 1u);
        } else if (ONE && c < CH && c * 64 + lane < P) {
            atomicOr(err, 2u);
        }
    }
    if constexpr (ONE) __syncthreads();
    if (wv == 0) scan_units(s_tot, E, lists, s_off, s_unit, s_cap);
    __syncthreads();
    // counts -> exclusive prefix over the segment's chunks; S threads (a power
    // of two, in one wave) share an expert's chunks
    {
        uint32_t S = CH;
        while (S > 1 && E * S > PERM_THREADS) S >>= 1;
        const uint32_t e = threadIdx.x / S, sg = threadIdx.x % S;
        const uint32_t Lc = CH / S, c0 = sg * Lc;
        uint32_t sum = 0;
        if (e < E)
            for (uint32_t c = c0; c < c0 + Lc; ++c) sum += s_cnt[e * CS + c];
        uint32_t inc = sum;
        for (uint32_t dlt = 1; dlt < S; dlt <<= 1) {
            const uint32_t o = __shfl_up(inc, dlt, S);
            if (sg >= dlt) inc += o;
        }
        if (e < E) {
            uint32_t run = s_off[e] + s_base[e] + inc - sum;
            for (uint32_t c = c0; c < c0 + Lc; ++c) {
                const uint32_t t = s_cnt[e * CS + c];
                s_cnt[e * CS + c] = run;
                run += t;
            }
        }
    }
    __syncthreads();
    uint32_t nbits = 1;
    while ((1u << nbits) < E) ++nbits;
#pragma unroll
    for (uint32_t k = 0; k < 2; ++k) {
        const uint32_t c = wv + k * NW, e = eid[k];
        const bool ok = e < E;
        uint64_t same = __ballot(ok);
        for (uint32_t b = 0; b < nbits; ++b) {
            const bool bit = (e >> b) & 1u;
            const uint64_t set = __ballot(ok && bit);
            same &= bit ? set : ~set;
        }
        const uint32_t rank = __popcll(same & ((1ull << lane) - 1ull));
        if (ok) sorted_pairs[s_cnt[e * CS + c] + rank] = (seg * CH + c) * 64 + lane;
    }
    if (seg == 0) write_units(s_off, s_unit, E, s_cap, lists);
}

// ---------------------------------------------------------------------------
// k_grouped_mm: for each unit (a pass of up to 64 pairs of an expert),
// out[pair][n] for one tile of its weight matrix: 128 rows of gate and of up
// (gate+up, SiLU fused) or 256 rows of down.  Block = 8 waves; wave w owns two
// 16-row MFMA subtiles (gate and up rows 16w.., or down rows 32w.. and
// 32w + 16..) and all m-tiles of the pass.  Serves rows with an odd number of
// groups, weights that are not 16-byte aligned, and grids of at most one block a
// CU (lds_weights); others take k_grouped_reg.
//
// The k dimension streams through two rings in LDS, filled by direct
// global->LDS loads (global_load_lds_dwordx4) so that nothing in flight holds
// registers:
//   weights      GM_SW stages of two 64-column groups: every wave brings its
//                32 rows x 64 bytes of codes (each row's 64 bytes in one
//                instruction: 32-byte pieces per row halve the stream rate)
//                and the rows' two fp16 scales;
//   activations  GM_SA stages of one group: the pass's rows (f16 hi and lo
//                planes), a share per wave.
// Body c (one group) waits for its stages, passes one barrier, requests
// activation stage c + 3 and then (even c) weight stage c/2 + 3, and computes:
// the weights, from HBM, then have five bodies before a wait covers them.  Each stage
// lives in its own __shared__ object, so the compiler can tell the in-flight
// fills from the stage being read; completion is awaited with an explicit
// vmcnt: every wave issues the same loads in the same order.
//
// v_mfma_f32_16x16x32_f16 operand layout: lane l holds A[l % 16][8 (l/16) + j]
// and B[8 (l/16) + j][l % 16] (j < 8) and receives D[4 (l/16) + i][l % 16].
// Inside a 64-column group, lane quarter q = l/16 of MFMA step s uses the
// physical columns 32 s + 8 q + j (both operands hold a lane's 8 columns in
// the order 0 2 4 6 1 3 5 7), as k_grouped_reg does: a pair's sums are the same
// bits in either kernel.  Weights enter as f16 (2c - 15)/8 (exact), so
// a group's MFMA sum times s_g is 15/60 of its dequantised dot product
// (kernels.metal:90-105, 140-145) and the epilogue is one FMA per output.
// LDS layouts (16-byte slots; XOR swizzles keep the fragment reads free of
// bank conflicts):
//   weights  subtile j of wave w: row n, slot (2 g + h) ^ (n >> 2 & 3) holds
//            bytes 16 h .. 16 h + 15 of group g of the stage;
//   acts     row r, slot x ^ (r & 15) = logical slot x = 8 plane + c8, i.e.
//            columns 8 c8 .. 8 c8 + 7 of the group in plane hi (0) or lo (1).
// ---------------------------------------------------------------------------
constexpr int GM_WAVES = 8;
constexpr int GM_SW = 4;                     // weight ring stages (two 64-column groups each)
constexpr int GM_SA = 4;                     // activation ring stages (one group each)
constexpr int GM_PASS = 64;                  // pair rows per pass (4 m-tiles)
constexpr uint32_t GM_ROWS_GU = 16 * GM_WAVES;   // gate (and up) rows per block
constexpr uint32_t GM_ROWS_DN = 32 * GM_WAVES;   // down rows per block

struct GmW {                                 // one weight stage: 2 groups of the block's rows
    uint8_t w[GM_WAVES * 2048];              // per wave: subtile j (1 KB) = 16 rows x 4 slots of 16 B
    uint32_t sc[GM_WAVES * 64];              // per wave: slot 32 g + 16 j + n holds the fp16 scale
};
struct GmA { uint8_t a[GM_PASS * 256]; };    // one activation stage: row = 16 slots (hi, lo) x 64 columns

#define SMOE_LDS_AS(p) ((__attribute__((address_space(3))) void*)(p))

// 8 codes (a word: byte b holds codes 2b (low nibble) and 2b + 1) -> 8 f16
// (c - 7.5) / 4 in the order 0 2 4 6 1 3 5 7.  A code shifted to bits 4..7 of
// a byte under the byte 0x4C is the f16 16 + c/4 (exponent 4, mantissa
// c << 4), one v_perm per two codes; 16 + c/4 - 17.875 = (c - 7.5)/4 is exact.
__device__ __forceinline__ half8_t q4_codes_to_f16(uint32_t v)
{
    const uint32_t E = (v << 4) & 0xF0F0F0F0u;    // even codes << 4
    const uint32_t O = v & 0xF0F0F0F0u;           // odd codes << 4
    const uint32_t K = 0x4C4C4C4Cu;
    u32x4_t r;
    r.x = __builtin_amdgcn_perm(K, E, 0x04010400u);   // codes 0, 2
    r.y = __builtin_amdgcn_perm(K, E, 0x04030402u);   // codes 4, 6
    r.z = __builtin_amdgcn_perm(K, O, 0x04010400u);   // codes 1, 3
    r.w = __builtin_amdgcn_perm(K, O, 0x04030402u);   // codes 5, 7
    const _Float16 b = static_cast<_Float16>(-17.875f);
    const half8_t bias = {b, b, b, b, b, b, b, b};
    return __builtin_bit_cast(half8_t, r) + bias;
}

__device__ __forceinline__ half8_t lds_half8(const uint8_t* p)
{
    const uint4 v = *reinterpret_cast<const uint4*>(__builtin_assume_aligned(p, 16));
    u32x4_t u;
    u.x = v.x; u.y = v.y; u.z = v.z; u.w = v.w;
    return __builtin_bit_cast(half8_t, u);
}

template <int N>
__device__ __forceinline__ void vm_wait()
{
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}
// the same, and this wave's LDS reads are done
template <int N>
__device__ __forceinline__ void vm_lds_wait()
{
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4));
}
__device__ __forceinline__ void mem_fence_compiler() { asm volatile("" ::: "memory"); }
__device__ __forceinline__ void gm_barrier()
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

template <bool GATE_UP, int MS>
__device__ __forceinline__ void grouped_mm_expert(
    const MoeDims& d, const LayerDesc& L, uint32_t e, uint32_t tile, uint32_t base, uint32_t M,
    const uint32_t* __restrict__ sorted_pairs, const uint16_t* __restrict__ a_hi, const uint16_t* __restrict__ a_lo,
    const float* __restrict__ a_scale, uint32_t a_row_div, float* __restrict__ out, uint32_t n_dim, uint32_t k_dim,
    GmW& w0, GmW& w1, GmW& w2, GmW& w3, GmA& a0, GmA& a1, GmA& a2, GmA& a3, uint32_t (&s_row)[GM_PASS],
    uint32_t (&s_pair)[GM_PASS])
{
    constexpr int AN = MS >= 3 ? 2 : 1;          // activation loads per wave and stage (4 rows each;
                                                 // at MS = 3 rows past the pass repeat its last row)
    constexpr int PASS = 16 * MS;
    const int lane = threadIdx.x & 63;
    const uint32_t wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t G = k_dim >> 6;
    const uint32_t m16 = lane & 15, q = lane >> 4;

    const uint8_t* blob = L.experts + static_cast<size_t>(e) * L.stride;
    const size_t row_bytes = k_dim >> 1;
    auto w_row = [&](uint32_t j, uint32_t n) -> uint32_t {
        const uint32_t r = GATE_UP ? tile * GM_ROWS_GU + 16 * wv + n : tile * GM_ROWS_DN + 32 * wv + 16 * j + n;
        return min(r, n_dim - 1);
    };
    auto w_mat = [&](uint32_t j) -> const uint8_t* { return blob + (GATE_UP ? (j ? L.off[2] : L.off[0]) : L.off[4]); };
    auto s_mat = [&](uint32_t j) -> const uint16_t* {
        return reinterpret_cast<const uint16_t*>(blob + (GATE_UP ? (j ? L.off[3] : L.off[1]) : L.off[5]));
    };
    // weight fill, instruction j: lane -> row n = lane / 4, physical slot p = lane & 3,
    // logical slot s = p ^ (n / 4 & 3) = 2 g + h: bytes 32 g + 16 h of the stage's 64
    const uint32_t fn = lane >> 2, fs = (lane & 3) ^ ((fn >> 2) & 3);
    const uint32_t fg = fs >> 1, fh = fs & 1;
    const uint8_t* w_src[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) w_src[j] = w_mat(j) + static_cast<size_t>(w_row(j, fn)) * row_bytes + 16 * fh;
    // scale fill: lane -> group g = lane / 32 of the stage, subtile (lane / 16) & 1, row lane & 15
    const uint32_t sg = lane >> 5, sj = (lane >> 4) & 1, sn = lane & 15;
    const uint16_t* s_src = s_mat(sj) + static_cast<size_t>(w_row(sj, sn)) * G;
    // (an odd G's last stage has one group: its second group re-reads group G - 1)
    auto issue_w = [&](GmW& S, uint32_t st) {
        const uint32_t g0 = 2 * st + fg, gs = 2 * st + sg;
#pragma unroll
        for (int j = 0; j < 2; ++j)
            __builtin_amdgcn_global_load_lds(w_src[j] + min(g0, G - 1) * 32, SMOE_LDS_AS(&S.w[wv * 2048 + j * 1024]),
                                             16, 0, 0);
        __builtin_amdgcn_global_load_lds(s_src + min(gs, G - 1), SMOE_LDS_AS(&S.sc[wv * 64]), 2, 0, 0);
    };
    // B fragment of this lane for group g of a stage, step stp: row m16, unit 4 stp + q (4 bytes) of the group
    uint32_t boff[2][2];
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int stp = 0; stp < 2; ++stp)
            boff[g][stp] = wv * 2048 + m16 * 64 + 16 * ((2 * g + stp) ^ ((m16 >> 2) & 3)) + 4 * q;
    // A fragment offsets of this lane inside an activation stage (m-tile ms adds 4096 bytes)
    uint32_t aoff[2][2];
#pragma unroll
    for (int stp = 0; stp < 2; ++stp)
#pragma unroll
        for (int pl = 0; pl < 2; ++pl) aoff[stp][pl] = m16 * 256 + 16 * ((8 * pl + 4 * stp + q) ^ m16);

    if (threadIdx.x < PASS) {
        const uint32_t p = sorted_pairs[base + min(threadIdx.x, M - 1)];
        s_pair[threadIdx.x] = p;
        s_row[threadIdx.x] = p / a_row_div;
    }
    __syncthreads();
    const uint16_t* a_src[AN];
#pragma unroll
    for (int u = 0; u < AN; ++u) {
        const uint32_t r = wv * 4 * AN + 4 * u + (lane >> 4);
        const uint32_t x = (lane & 15) ^ (r & 15);
        const uint32_t srow = s_row[min(r, static_cast<uint32_t>(PASS - 1))];
        a_src[u] = ((x >> 3) ? a_lo : a_hi) + static_cast<size_t>(srow) * k_dim + 8 * (x & 7);
    }
    auto issue_a = [&](GmA& S, uint32_t c) {
#pragma unroll
        for (int u = 0; u < AN; ++u)
            __builtin_amdgcn_global_load_lds(a_src[u] + c * 64, SMOE_LDS_AS(&S.a[(wv * 4 * AN + 4 * u) * 256]), 16,
                                             0, 0);
    };

    f32x4_t acc[MS][2];
#pragma unroll
    for (int ms = 0; ms < MS; ++ms)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[ms][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    // Issue order of the loop: body c issues the activation stage c + 3 and then the
    // weight stage c / 2 + 3 (if c is even).  The prologue replays bodies -6 .. -1.
    const uint32_t NWS = (G + 1) / 2;        // weight stages
    if (0 < NWS) issue_w(w0, 0);
    if (1 < NWS) issue_w(w1, 1);
    if (0 < G) issue_a(a0, 0);
    if (1 < G) issue_a(a1, 1);
    if (2 < NWS) issue_w(w2, 2);
    if (2 < G) issue_a(a2, 2);
    mem_fence_compiler();

    auto body = [&](uint32_t c, GmW& W, uint32_t g, GmW& WN, GmA& A, GmA& AN_) {
        // A(c) was the first load of body c - 3; after it came the weight stage of body
        // c - 3 when c - 3 is even, A(c + 1), A(c + 2) and the weight stage of the even
        // one of bodies c - 2, c - 1 ((c + 4 + (c & 1)) / 2, the later of the two).  When
        // all of those were issued, 2 AN + 3 (even c) or 2 AN + 6 (odd c) loads may still
        // be pending; near the end fewer were, and the wait covers everything.
        if (c + 2 < G && (c + 4 + (c & 1)) / 2 < NWS) {
            if (g) vm_wait<2 * AN + 6>();
            else vm_wait<2 * AN + 3>();
        } else {
            vm_wait<0>();
        }
        gm_barrier();
        if (c + 3 < G) issue_a(AN_, c + 3);
        if (g == 0 && c / 2 + 3 < NWS) issue_w(WN, c / 2 + 3);
        mem_fence_compiler();
        half8_t b[2][2];
        float sc[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
#pragma unroll
            for (int stp = 0; stp < 2; ++stp)
                b[j][stp] = q4_codes_to_f16(*reinterpret_cast<const uint32_t*>(&W.w[boff[g][stp] + 1024 * j]));
            sc[j] = f16_bits_to_f32(static_cast<uint16_t>(W.sc[wv * 64 + 32 * g + 16 * j + m16]));
        }
#pragma unroll
        for (int ms = 0; ms < MS; ++ms) {
            half8_t xa[2][2];
#pragma unroll
            for (int stp = 0; stp < 2; ++stp)
#pragma unroll
                for (int pl = 0; pl < 2; ++pl) xa[stp][pl] = lds_half8(A.a + ms * 4096 + aoff[stp][pl]);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                f32x4_t t = {0.f, 0.f, 0.f, 0.f};
                t = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[0][0], b[j][0], t, 0, 0, 0);
                t = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[0][1], b[j][0], t, 0, 0, 0);
                t = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[1][0], b[j][1], t, 0, 0, 0);
                t = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[1][1], b[j][1], t, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[ms][j][i] = fmaf(sc[j], t[i], acc[ms][j][i]);
            }
        }
        mem_fence_compiler();
    };
    for (uint32_t c = 0; c < G; c += 8) {
        body(c, w0, 0, w3, a0, a3);
        if (c + 1 < G) body(c + 1, w0, 1, w3, a1, a0);
        if (c + 2 < G) body(c + 2, w1, 0, w0, a2, a1);
        if (c + 3 < G) body(c + 3, w1, 1, w0, a3, a2);
        if (c + 4 < G) body(c + 4, w2, 0, w1, a0, a3);
        if (c + 5 < G) body(c + 5, w2, 1, w1, a1, a0);
        if (c + 6 < G) body(c + 6, w3, 0, w2, a2, a1);
        if (c + 7 < G) body(c + 7, w3, 1, w2, a3, a2);
    }
#pragma unroll
    for (int ms = 0; ms < MS; ++ms) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t m = 16 * ms + 4 * q + i;
            if (m >= M) continue;
            const float rs = a_scale[s_row[m]] * (8.0f / 15.0f);   // weights are (2c - 15) / 8
            float* o = out + static_cast<size_t>(s_pair[m]) * n_dim;
            if (GATE_UP) {
                const uint32_t n = tile * GM_ROWS_GU + 16 * wv + m16;
                if (n < n_dim) {
                    const float v0 = acc[ms][0][i] * rs, v1 = acc[ms][1][i] * rs;
                    o[n] = (v0 * (1.0f / (1.0f + expf(-v0)))) * v1;
                }
            } else {
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const uint32_t n = tile * GM_ROWS_DN + 32 * wv + 16 * j + m16;
                    if (n < n_dim) o[n] = acc[ms][j][i] * rs;
                }
            }
        }
    }
}

// block b of a grid over units x n_tiles -> the unit's record (its own slot,
// see write_units) and the tile: XCD b mod 8, tile by tile of a unit
__device__ __forceinline__ uint4 unit_of_block(const uint4* __restrict__ units, uint32_t n_tiles, uint32_t& tile)
{
    const uint32_t b = blockIdx.x, jb = b >> 3;
    tile = jb % n_tiles;
    return units[8u * (jb / n_tiles) + (b & 7u)];
}

template <bool GATE_UP>
__global__ __launch_bounds__(GM_WAVES * WAVE, 1)
void k_grouped_mm(MoeDims d, LayerDesc L, const uint4* __restrict__ units, const uint32_t* __restrict__ sorted_pairs, const uint16_t* __restrict__ a_hi,
                  const uint16_t* __restrict__ a_lo, const float* __restrict__ a_scale, uint32_t a_row_div,
                  float* __restrict__ out, uint32_t n_dim, uint32_t k_dim, uint32_t n_tiles)
{
    __shared__ __align__(16) GmW w0, w1, w2, w3;
    __shared__ __align__(16) GmA a0, a1, a2, a3;
    __shared__ uint32_t s_row[GM_PASS];
    __shared__ uint32_t s_pair[GM_PASS];
    uint32_t tile;
    const uint4 rec = unit_of_block(units, n_tiles, tile);
    if (rec.z == 0) return;
    const uint32_t rows = rec.x >> 16;
    auto go = [&](auto ms) {
        grouped_mm_expert<GATE_UP, decltype(ms)::value>(d, L, rec.x & 0xFFFFu, tile, rec.y, rec.z, sorted_pairs, a_hi, a_lo, a_scale,
                                                        a_row_div, out, n_dim, k_dim, w0, w1, w2, w3, a0, a1, a2, a3,
                                                        s_row, s_pair);
    };
    if (rows == 16) go(std::integral_constant<int, 1>{});
    else if (rows == 32) go(std::integral_constant<int, 2>{});
    else if (rows == 48) go(std::integral_constant<int, 3>{});
    else go(std::integral_constant<int, 4>{});
}

// ---------------------------------------------------------------------------
// grouped_reg: the grouped products with the weights streamed into registers:
// each weight row belongs to one wave, so plain loads need neither LDS nor a
// barrier for them.  Blocks of 4 waves x 64 weight rows (four 16-row subtiles
// a wave; gate/up: 32 gate rows and the same 32 up rows), two blocks per CU:
// every activation fragment read from LDS feeds four subtiles, and the two
// blocks of a CU pass their barriers independently, so one block's MFMAs
// overlap the other's conversion.  Needs an even number of groups (a stage's
// two scales are one dword).
//   stage    two 64-column groups; gd_depth stages are requested ahead of the one
//            that is computed: their codes in registers, their activation rows in
//            a ring in LDS, one counted wait and one barrier per stage.  As
//            compiled the ring does not stay that full: the loop's exits after
//            each stage let the registers of the codes meet at its latch, where
//            the compiler waits for every load in flight, once in gd_depth stages
//            (not where that is one), and the waits that it adds before the codes'
//            uses count without the rows' loads, which it does not see, so they
//            are stricter than the counted ones;
//   weights  up to two m-tiles a unit (HBM-bound): a load takes 128 bytes of 8
//            rows, the codes of two stages, marked non-temporal (each weight
//            line is read once).  Whole lines set the stream's rate: the loads
//            alone run 805 MB of gate/up in 153 us as 64 bytes of 16 rows (194
//            non-temporal), 141 as whole lines, 125 (6.4 TB/s) as whole lines
//            non-temporal.  Lane l loads row l & 7, unit l >> 3; a rotation by
//            8 in each 16 lanes, v_permlane32_swap and v_permlane16_swap leave
//            quad q = l >> 4, MFMA step s the 8-column unit 4 s + q of each
//            group, row l & 15.  More m-tiles (bound by the matrix cores; their
//            registers hold fewer stages): 64 bytes of 16 rows, lane l row
//            l & 15, bytes 16 (l >> 4) .. + 15, and the two swaps leave the
//            same units: a pair's sums do not depend on its unit's size;
//   acts     [plane][row][16 units of 8 columns], unit x of row r in slot
//            x ^ (r & 15): conflict-free for the fragment reads (units 4 s + q
//            of rows 0 .. 15), filled by direct loads (4 rows x 256 bytes each)
//            issued from inline asm: the compiler does not track them, so it does
//            not drain them before the reads of another stage's rows;
//   scales   one load of eight groups of the wave's rows instead of a load per
//            row and stage, passed across the wave (ds_bpermute).
//   MFMA     the four products of a group (hi and lo of two steps) accumulate
//            in one register set per subtile; the four subtiles' chains run
//            interleaved, the next m-tile's fragments are read during them, and
//            the sums are scaled into the accumulators during the next
//            m-tile's chains.
// Nothing stands between a block's start and its weights but its record; the
// pairs, the rows' addresses and their scales stay in registers.
// Measured against the kernels before it (weights of gate/up through LDS, 8
// waves and one block per CU; passes of at most 736 tokens): 4096 tokens of the
// 30B shape gate/up 700 -> 396 us (1.08 PFLOP/s of f16 products; a library f16
// GEMM reaches 1.19 on the same card), down 407 -> 229; 512 tokens gate/up 97 ->
// 82, down 54 -> 45; 64 tokens of the 235B shape gate/up 248 -> 186 (4.6 TB/s;
// one stage in flight and 64-byte loads: 202), down 125 -> 106 (115).  Three
// blocks per CU with 168 registers: no faster (spills).
// ---------------------------------------------------------------------------
constexpr int GD_WAVES = 4;
constexpr int GD_SUB = 4;                                  // 16-row subtiles a wave
constexpr uint32_t GD_ROWS = 16 * GD_SUB * GD_WAVES;       // weight rows per block
constexpr int GD_NT = 2;                                   // the loads' non-temporal bit
constexpr uint32_t GD_LDS = 80 * 1024;                     // the activation ring: half of a CU's LDS
// stages in flight: what the ring (DP + 1 stages of 8 KB an m-tile) and the registers hold
constexpr int gd_depth(int ms) { return ms <= 2 ? 4 : ms == 3 ? 2 : 1; }

__device__ __forceinline__ uint32_t lds_addr(const void* p)
{
    return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) void*)p));
}
// a resource over `bytes` of weights at p (wave-uniform): loads past it return 0
__device__ __forceinline__ __amdgpu_buffer_rsrc_t weight_rsrc(const void* p, uint32_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, static_cast<int>(bytes), 0x00020000);
}
// lane l's 16 bytes at base + off (off per lane) land at LDS byte address lds + 16 l
__device__ __forceinline__ void dma16(const void* base, uint32_t off, uint32_t lds)
{
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds)
                 : "memory", "m0");
}

// The np <= 16 MS pairs from sorted_pairs[first] on, all of expert e; one tile of GD_ROWS weight rows.
template <bool GATE_UP, int MS>
__device__ __forceinline__ void grouped_reg_expert(
    const LayerDesc& L, uint32_t e, uint32_t tile, uint32_t first, uint32_t np,
    const uint32_t* __restrict__ sorted_pairs, const uint16_t* __restrict__ a_hi, const uint16_t* __restrict__ a_lo,
    const float* __restrict__ a_scale, uint32_t a_row_div, float* __restrict__ out, uint32_t n_dim, uint32_t k_dim,
    uint8_t* abuf)
{
    constexpr int PASS = 16 * MS;
    constexpr int DP = gd_depth(MS);             // stages in flight
    // QUAD: the codes of two stages in one load, 128 bytes of 8 rows (a whole
    // line a row: the stream's rate hangs on it); else 64 bytes of 16 rows
    constexpr bool QUAD = DP == 4;
    constexpr int WL = QUAD ? 2 * GD_SUB : GD_SUB, WD = QUAD ? DP / 2 : DP;
    constexpr uint32_t PLANE = PASS * 256, STAGE = 2 * PLANE;
    static_assert((DP + 1) * STAGE <= GD_LDS, "the ring fits");
    const int lane = threadIdx.x & 63;
    const uint32_t wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t G = k_dim >> 6, NST = G / 2;
    const uint32_t m16 = lane & 15, q = lane >> 4;
    const uint32_t pair = sorted_pairs[first + min(static_cast<uint32_t>(lane), np - 1)];

    // codes and scales through buffer resources: a scalar base and one offset
    // register a subtile (64-bit addresses took 16 registers more and spilled)
    const uint8_t* blob = L.experts + static_cast<size_t>(e) * L.stride;
    constexpr int NM = GATE_UP ? 2 : 1, SM = GD_SUB / NM;   // matrices, subtiles of each
    const uint32_t w_bytes = n_dim * (k_dim >> 1);
    const uint8_t* w_mat[NM];
    __amdgpu_buffer_rsrc_t s_mat[NM];
#pragma unroll
    for (int i = 0; i < NM; ++i) {
        const int o = GATE_UP ? 2 * i : 4;
        w_mat[i] = blob + L.off[o];
        s_mat[i] = weight_rsrc(blob + L.off[o + 1], n_dim * G * 2);
    }
    // gate/up: subtiles 0, 1 are 32 gate rows, 2, 3 the same rows of up (n_dim is
    // a multiple of 64: a subtile past the end is a repeat of the last one)
    const uint32_t row_w = tile * (GD_ROWS / NM) + 16 * SM * wv, row_bytes = k_dim >> 1;
    auto row_j = [&](int j) { return min(row_w + 16 * (j % SM), n_dim - 16); };
    uint32_t w_off[SM];                          // QUAD: w_off[0] only, the subtile is a scalar offset
#pragma unroll
    for (int j = 0; j < SM; ++j)
        w_off[j] = QUAD ? (lane & 7) * row_bytes + 16 * (lane >> 3) : (row_j(j) + m16) * row_bytes + 16 * q;
    // scales: lane l loads eight groups of the wave's row l (% 32) at once
    // (every load instruction costs the CU a request slot whatever its width:
    // one load per four pairs of groups instead of four per pair); the lanes
    // that use them fetch them across the wave
    const uint32_t s_off = min(row_w + (lane & (16 * SM - 1)), n_dim - 1) * G * 2;
    u32x4_t sc_next[NM], sc_cur[NM];             // scales of eight groups: the next ones, the current ones
    auto issue_s = [&](uint32_t piece) {
#pragma unroll
        for (int i = 0; i < NM; ++i) sc_next[i] = __builtin_amdgcn_raw_buffer_load_b128(s_mat[i], s_off, 16 * piece, 0);
    };
    // (past the last stage the resource is empty: the load returns 0 and moves
    // nothing, and every stage issues the same number of loads)
    u32x4_t wr[WD][WL];                          // the codes in flight
    auto issue_w = [&](u32x4_t (&W)[WL], uint32_t k) {
        if constexpr (QUAD) {
            const bool in = 2 * k < NST;
            // (an odd last stage: both halves of the lanes load it)
            const uint32_t off = 2 * k + 1 < NST ? w_off[0] : w_off[0] - 2 * (lane & 32);
#pragma unroll
            for (int j = 0; j < WL; ++j)
                W[j] = __builtin_amdgcn_raw_buffer_load_b128(
                    weight_rsrc(w_mat[j / 2 / SM], in ? w_bytes : 0u), off,
                    in ? (row_j(j / 2) + 8 * (j & 1)) * row_bytes + 128 * k : 0u, GD_NT);
        } else {
            const bool in = k < NST;
#pragma unroll
            for (int j = 0; j < WL; ++j)
                W[j] = __builtin_amdgcn_raw_buffer_load_b128(weight_rsrc(w_mat[j / SM], in ? w_bytes : 0u),
                                                             w_off[j % SM], in ? 64 * k : 0u, 0);
        }
    };
    issue_s(0);
#pragma unroll
    for (int i = 0; i < WD; ++i) issue_w(wr[i], i);

    // lane l: the row of pair l of the unit, and its scale
    const uint32_t arow = GATE_UP ? pair / a_row_div : pair;
    const float ascale = a_scale[arow];
    // activation fill: waves 0, 1 the hi plane, 2, 3 the lo plane, 2 MS loads of 4 rows each
    const uint16_t* plane = wv >= 2 ? a_lo : a_hi;
    const uint32_t row0 = (wv & 1) * 8 * MS;
    uint32_t a_off[2 * MS];
#pragma unroll
    for (int u = 0; u < 2 * MS; ++u) {
        const uint32_t r = row0 + 4 * u + q;
        a_off[u] = (__builtin_amdgcn_ds_bpermute(4 * r, arow) * k_dim + 8 * (m16 ^ (r & 15))) * 2;
    }
    const uint32_t a_dst = lds_addr(abuf) + (wv >> 1) * PLANE + row0 * 256;
    auto issue_a = [&](uint32_t slot, uint32_t st) {
        const uint8_t* src = reinterpret_cast<const uint8_t*>(plane) + 256 * st;
#pragma unroll
        for (int u = 0; u < 2 * MS; ++u) dma16(src, a_off[u], a_dst + slot * STAGE + u * 1024);
    };
    mem_fence_compiler();
#pragma unroll
    for (int i = 0; i < DP; ++i)
        if (static_cast<uint32_t>(i) < NST) issue_a(i, i);
    mem_fence_compiler();

    // fragment of group g, step s of this lane (unit 4 s + q): 16 bytes at aoff[g][s] (m-tile ms: + 4096 ms; lo plane: + PLANE)
    uint32_t aoff[2][2];
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int stp = 0; stp < 2; ++stp)
            aoff[g][stp] = m16 * 256 + 16 * ((8 * g + 4 * stp + q) ^ m16);

    f32x4_t acc[MS][GD_SUB];
#pragma unroll
    for (int ms = 0; ms < MS; ++ms)
#pragma unroll
        for (int j = 0; j < GD_SUB; ++j) acc[ms][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    uint32_t slot = 0;                           // st % (DP + 1): the ring slot of stage st
    uint32_t gw[QUAD ? 2 : 1][GD_SUB][2][2];     // [stage of a quad][subtile][group][MFMA step]
    auto stage = [&](auto dc, uint32_t st) {
        constexpr int D = decltype(dc)::value;   // st % DP
        // What may still be pending when stage st's codes and rows are needed:
        // what stages st - DP + 1 .. st - 1 issued, each its rows (2 MS loads;
        // none past the end) before its codes.  The first DP stages' codes all
        // went before their rows.
        constexpr bool EVEN = !QUAD || D % 2 == 0;
        constexpr int A_N = 2 * MS * (DP - 1), W_N = QUAD ? WL * (EVEN ? 1 : 2) : WL * (DP - 1);
        if (st + DP > NST) {
            if (st < DP) vm_lds_wait<0>();
            else vm_lds_wait<W_N>();
        } else if (st < DP) {
            vm_lds_wait<A_N + (QUAD ? WL * ((D + 1) / 2) : WL * D)>();
        } else {
            vm_lds_wait<A_N + W_N>();
        }
        gm_barrier();
        if constexpr (!QUAD) {
#pragma unroll
            for (int j = 0; j < GD_SUB; ++j) {
                const auto u = __builtin_amdgcn_permlane32_swap(wr[D][j][0], wr[D][j][2], false, false);
                const auto v = __builtin_amdgcn_permlane32_swap(wr[D][j][1], wr[D][j][3], false, false);
#pragma unroll
                for (int g = 0; g < 2; ++g) {
                    const auto r = __builtin_amdgcn_permlane16_swap(u[g], v[g], false, false);
                    gw[0][j][g][0] = r[0];
                    gw[0][j][g][1] = r[1];
                }
            }
        } else if constexpr (EVEN) {
            // lane bits 5 4 3 | 2 1 0 hold group, group, half of the group | row,
            // the registers row bit 3 (x, y) and the word of the half.  Half and
            // row bit 3 change places, then the group's bits and the word's:
            // quad q has word q of either half of every group, row m16.
#pragma unroll
            for (int j = 0; j < GD_SUB; ++j) {
                uint32_t hw[2][4];
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const int x = wr[D / 2][2 * j][w], y = wr[D / 2][2 * j + 1][w];
                    hw[0][w] = __builtin_amdgcn_update_dpp(x, y, 0x128, 0xF, 0xC, false);   // row_ror:8
                    hw[1][w] = __builtin_amdgcn_update_dpp(y, x, 0x128, 0xF, 0x3, false);
                }
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const auto u = __builtin_amdgcn_permlane32_swap(hw[h][0], hw[h][2], false, false);
                    const auto v = __builtin_amdgcn_permlane32_swap(hw[h][1], hw[h][3], false, false);
#pragma unroll
                    for (int p = 0; p < 2; ++p) {
                        const auto r = __builtin_amdgcn_permlane16_swap(u[p], v[p], false, false);
                        gw[p][j][0][h] = r[0];
                        gw[p][j][1][h] = r[1];
                    }
                }
            }
        }
        if (st % 4 == 0) {
#pragma unroll
            for (int i = 0; i < NM; ++i) sc_cur[i] = sc_next[i];
            issue_s(min(st / 4 + 1, (NST - 1) / 4));
        }
        // every wave is past stage st - 1: its slot takes stage st + DP
        if (st + DP < NST) issue_a(slot == 0 ? DP : slot - 1, st + DP);
        if constexpr (!QUAD) issue_w(wr[D], st + DP);
        else if constexpr (EVEN) issue_w(wr[D / 2], (st + DP) / 2);
        mem_fence_compiler();
        __builtin_amdgcn_sched_barrier(0);
        uint32_t sc2[GD_SUB];                    // the two groups' fp16 scales
#pragma unroll
        for (int j = 0; j < GD_SUB; ++j)
            sc2[j] = __builtin_amdgcn_ds_bpermute(4 * (16 * (j % SM) + m16), sc_cur[j / SM][0]);
#pragma unroll
        for (int i = 0; i < NM; ++i) {
            sc_cur[i][0] = sc_cur[i][1];
            sc_cur[i][1] = sc_cur[i][2];
            sc_cur[i][2] = sc_cur[i][3];
        }
        const uint8_t* A = abuf + slot * STAGE;
        slot = slot == DP ? 0 : slot + 1;
        // fragment c (step c / 2, plane c & 1) of m-tile k % MS of group k / MS
        half8_t xa[4];
        auto load_a = [&](int k, int c) {
            xa[c] = lds_half8(A + (c & 1) * PLANE + (k % MS) * 4096 + aoff[k / MS][c >> 1]);
        };
        // The sched_barriers pin the order (left to itself the compiler reads
        // each fragment right before its use and runs the chains one after
        // the other, waiting out every latency).
#pragma unroll
        for (int c = 0; c < 4; ++c) load_a(0, c);
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            f32x4_t t[GD_SUB];
            half8_t b[GD_SUB][2];
            float sc[GD_SUB];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < GD_SUB; ++j) {
                b[j][0] = q4_codes_to_f16(gw[QUAD ? D % 2 : 0][j][g][0]);
                sc[j] = f16_bits_to_f32(static_cast<uint16_t>(g ? sc2[j] >> 16 : sc2[j]));
            }
            auto scale_in = [&](int ms, int j) {
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[ms][j][i] = fmaf(sc[j], t[j][i], acc[ms][j][i]);
            };
#pragma unroll
            for (int ms = 0; ms < MS; ++ms) {
                const int k = g * MS + ms;
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int c = 0; c < 4; ++c) {
#pragma unroll
                    for (int j = 0; j < GD_SUB; ++j) {
                        const f32x4_t z = {0.f, 0.f, 0.f, 0.f};
                        if (c == 0 && ms > 0) scale_in(ms - 1, j);
                        t[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[c], b[j][c >> 1], c ? t[j] : z, 0, 0, 0);
                    }
                    if (ms == 0 && c < 2) {
                        b[2 * c][1] = q4_codes_to_f16(gw[QUAD ? D % 2 : 0][2 * c][g][1]);
                        b[2 * c + 1][1] = q4_codes_to_f16(gw[QUAD ? D % 2 : 0][2 * c + 1][g][1]);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    if (k + 1 < 2 * MS) load_a(k + 1, c);
                }
            }
#pragma unroll
            for (int j = 0; j < GD_SUB; ++j) scale_in(MS - 1, j);
        }
        mem_fence_compiler();
    };
    for (uint32_t st = 0;;) {
        stage(std::integral_constant<int, 0>{}, st);
        if (++st >= NST) break;
        if constexpr (DP > 1) {
            stage(std::integral_constant<int, 1>{}, st);
            if (++st >= NST) break;
        }
        if constexpr (DP > 2) {
            stage(std::integral_constant<int, 2 % DP>{}, st);
            if (++st >= NST) break;
        }
        if constexpr (DP > 3) {
            stage(std::integral_constant<int, 3 % DP>{}, st);
            if (++st >= NST) break;
        }
    }
#pragma unroll
    for (int ms = 0; ms < MS; ++ms) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t m = 16 * ms + 4 * q + i;
            const uint32_t p = __builtin_amdgcn_ds_bpermute(4 * m, pair);
            const float as = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(4 * m, __builtin_bit_cast(int, ascale)));
            if (m >= np) continue;
            const float rs = as * (8.0f / 15.0f);   // weights are (2c - 15) / 8
            float* o = out + static_cast<size_t>(p) * n_dim;
            if constexpr (GATE_UP) {
#pragma unroll
                for (int j = 0; j < GD_SUB / 2; ++j) {
                    const uint32_t n = tile * (GD_ROWS / 2) + 8 * GD_SUB * wv + 16 * j + m16;
                    const float v0 = acc[ms][j][i] * rs, v1 = acc[ms][j + GD_SUB / 2][i] * rs;
                    if (n < n_dim) o[n] = (v0 * (1.0f / (1.0f + expf(-v0)))) * v1;
                }
            } else {
#pragma unroll
                for (int j = 0; j < GD_SUB; ++j) {
                    const uint32_t n = tile * GD_ROWS + 16 * GD_SUB * wv + 16 * j + m16;
                    if (n < n_dim) o[n] = acc[ms][j][i] * rs;
                }
            }
        }
    }
}

template <bool GATE_UP>
__global__ __launch_bounds__(GD_WAVES * WAVE, 2)
void k_grouped_reg(MoeDims d, LayerDesc L, const uint4* __restrict__ units,
                   const uint32_t* __restrict__ sorted_pairs, const uint16_t* __restrict__ a_hi,
                   const uint16_t* __restrict__ a_lo, const float* __restrict__ a_scale, uint32_t a_row_div,
                   float* __restrict__ out, uint32_t n_dim, uint32_t k_dim, uint32_t n_tiles)
{
    __shared__ __align__(16) uint8_t abuf[GD_LDS];
    uint32_t tile;
    const uint4 rec = unit_of_block(units, n_tiles, tile);
    if (rec.z == 0) return;
    const uint32_t rows = rec.x >> 16;
    auto go = [&](auto ms) {
        grouped_reg_expert<GATE_UP, decltype(ms)::value>(L, rec.x & 0xFFFFu, tile, rec.y, rec.z, sorted_pairs, a_hi,
                                                         a_lo, a_scale, a_row_div, out, n_dim, k_dim, abuf);
    };
    if (rows == 16) go(std::integral_constant<int, 1>{});
    else if (rows == 32) go(std::integral_constant<int, 2>{});
    else if (rows == 48) go(std::integral_constant<int, 3>{});
    else go(std::integral_constant<int, 4>{});
}

// ---------------------------------------------------------------------------
// k_combine_pairs: hidden[t][col] += sum_r w[t k + r] * y[(t k + r)][col], in
// rank order (the scatter-add of prefill.cpp:380-385 then :446-451).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256)
void k_combine_pairs(const float* __restrict__ y, const float* __restrict__ w, uint32_t K, uint32_t D,
                     float* __restrict__ hidden)
{
    // 4 columns per thread, the K rank rows of token t summed in rank order (one
    // load at a time per thread: the many resident waves hide the latency; loading
    // all K first measured no faster)
    const uint32_t t = blockIdx.y, col = (blockIdx.x * 256 + threadIdx.x) * 4;
    if (col >= D) return;
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    for (uint32_t r = 0; r < K; ++r) {
        const size_t p = static_cast<size_t>(t) * K + r;
        const float wr = w[p];
        const float4 v = load_f4(y + p * D + col);
        acc.x = fmaf(wr, v.x, acc.x);
        acc.y = fmaf(wr, v.y, acc.y);
        acc.z = fmaf(wr, v.z, acc.z);
        acc.w = fmaf(wr, v.w, acc.w);
    }
    float4* h = reinterpret_cast<float4*>(hidden + static_cast<size_t>(t) * D + col);
    const float4 o = *h;
    *h = make_float4(o.x + acc.x, o.y + acc.y, o.z + acc.z, o.w + acc.w);
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
template <int CPL, int TB, int ES = 1>
static hipError_t route_c(const MoeDims& d, const LayerDesc& L, const float* hidden, uint32_t T, uint16_t* x_hi,
                          uint16_t* x_lo, float* x_sc, uint32_t* ids, float* w, float* logits, uint32_t* counters,
                          hipStream_t s)
{
    const dim3 grid(((T + TB - 1) / TB) * ES), block(ROUTE_WAVES * WAVE);
    if (d.E <= 128)
        launch_kernel(k_route<CPL, TB, 2, ES>, grid, block, s, d, L, hidden, T, x_hi, x_lo, x_sc, ids, w,
                      logits, counters);
    else
        launch_kernel(k_route<CPL, TB, 8, ES>, grid, block, s, d, L, hidden, T, x_hi, x_lo, x_sc, ids, w,
                      logits, counters);
    return hipGetLastError();
}

hipError_t launch_route(const MoeDims& d, const LayerDesc& L, const float* hidden, uint32_t T, uint16_t* x_hi,
                        uint16_t* x_lo, float* x_sc, uint32_t* ids, float* w, float* logits, uint32_t* counters,
                        hipStream_t s)
{
    if (d.E > SMOE_TOPK_MAX_N || d.K > SMOE_TOPK_MAX_K || d.D % 64 || T == 0) return hipErrorInvalidValue;
    const uint32_t cpl = (d.D / 32 + WAVE - 1) / WAVE;
    // tokens per block: as few as give at most one block per CU (each block
    // reads the whole router matrix from L2 once, and a second round of blocks
    // costs as much as the first: 384 tokens of the 30B shape 24.8 us with one
    // token a block, 16.9 with two, 400 of the 235B shape 42.9 and 31), at most what the registers of a chunk per
    // lane allow.  Under 128 tokens (one per block) the router
    // rows of a token are split over 4 blocks (needs E <= 128: 4 rows a wave).
    const uint32_t cus = 256;
    const uint32_t tb = T > 2 * cus ? 4 : T > cus ? 2 : 1;
    const bool split = T < 128 && d.E <= 128 && logits && counters;
    if (cpl == 1) {
        if (tb == 4) return route_c<1, 4>(d, L, hidden, T, x_hi, x_lo, x_sc, ids, w, logits, counters, s);
        if (tb == 2) return route_c<1, 2>(d, L, hidden, T, x_hi, x_lo, x_sc, ids, w, logits, counters, s);
        if (split) return route_c<1, 1, 4>(d, L, hidden, T, x_hi, x_lo, x_sc, ids, w, logits, counters, s);
        return route_c<1, 1>(d, L, hidden, T, x_hi, x_lo, x_sc, ids, w, logits, counters, s);
    }
    if (cpl == 2) {
        if (tb >= 2) return route_c<2, 2>(d, L, hidden, T, x_hi, x_lo, x_sc, ids, w, logits, counters, s);
        if (split) return route_c<2, 1, 4>(d, L, hidden, T, x_hi, x_lo, x_sc, ids, w, logits, counters, s);
        return route_c<2, 1>(d, L, hidden, T, x_hi, x_lo, x_sc, ids, w, logits, counters, s);
    }
    if (cpl <= 4) return route_c<4, 1>(d, L, hidden, T, x_hi, x_lo, x_sc, ids, w, logits, counters, s);
    return hipErrorInvalidValue;
}

hipError_t launch_split_rows(const float* src, uint32_t rows, uint32_t cols, uint16_t* hi, uint16_t* lo,
                             float* scale, hipStream_t s)
{
    if (cols % 64 || rows == 0) return hipErrorInvalidValue;
    const uint32_t blocks = std::min<uint32_t>((rows + 3) / 4, 8192u);
    launch_kernel(k_split_rows, dim3(blocks), dim3(256), s, src, rows, cols, hi, lo, scale);
    return hipGetLastError();
}

// what k_permute allocates: the count table's odd row stride and the unit
// offsets add at most 3 E + 2 words to permute_lds_bytes (which bounds the batch)
static size_t permute_lds_alloc(uint32_t P, uint32_t E)
{
    const size_t CS = ((P + 63) / 64) | 1u;
    return (CS * E + 5 * size_t(E) + 3) * sizeof(uint32_t);
}

hipError_t launch_permute(const uint32_t* ids, const float* w, uint32_t P, uint32_t K, uint32_t E, uint32_t* offsets,
                          uint32_t* sorted_pairs, uint32_t* sorted_tokens, float* sorted_w, uint32_t* union_ids,
                          uint32_t* union_size, const UnitLists& lists, uint32_t* err, hipStream_t s)
{
    if (P == 0 || E == 0 || permute_lds_bytes(P, E) > PERMUTE_MAX_LDS) return hipErrorInvalidValue;
    const size_t lds = permute_lds_alloc(P, E);
    launch_kernel_lds(k_permute, dim3(1), dim3(PERM_THREADS), static_cast<uint32_t>(lds), s, ids, w, P, K, E,
                      offsets, sorted_pairs, sorted_tokens, sorted_w, union_ids, union_size, lists, err);
    return hipGetLastError();
}

hipError_t launch_permute_seg(const uint32_t* ids, uint32_t P, uint32_t E, uint32_t* sorted_pairs,
                              const UnitLists& lists, uint32_t* seg_cnt, uint32_t* err, hipStream_t s)
{
    if (P == 0 || E == 0 || E > SMOE_TOPK_MAX_N || !lists.units) return hipErrorInvalidValue;
    const uint32_t nseg = perm_segments(P, E);
    const uint32_t lds = (E * (perm_seg_chunks(E) | 1u) + 5 * E + 3) * static_cast<uint32_t>(sizeof(uint32_t));
    if (nseg == 1) {
        launch_kernel_lds(k_perm_scatter<true>, dim3(1), dim3(PERM_THREADS), lds, s, ids, P, E, seg_cnt,
                          sorted_pairs, lists, err);
        return hipGetLastError();
    }
    launch_kernel(k_perm_count, dim3(nseg), dim3(PERM_THREADS), s, ids, P, E, seg_cnt, err);
    launch_kernel_lds(k_perm_scatter<false>, dim3(nseg), dim3(PERM_THREADS), lds, s, ids, P, E, seg_cnt,
                      sorted_pairs, lists, err);
    return hipGetLastError();
}

// k_grouped_reg needs an even number of 64-column groups and its 16-byte
// weight loads; other layers take k_grouped_mm
static bool reg_supported(const LayerDesc& L, uint32_t k_dim)
{
    bool ok = k_dim % 128 == 0 && reinterpret_cast<uintptr_t>(L.experts) % 16 == 0 && L.stride % 16 == 0;
    for (int i = 0; i < 6; ++i) ok = ok && L.off[i] % 16 == 0;
    return ok;
}

template <bool GATE_UP>
static hipError_t launch_grouped(const MoeDims& d, const LayerDesc& L, uint32_t P, const UnitLists& lists,
                                 const uint32_t* sorted_pairs, const uint16_t* a_hi,
                                 const uint16_t* a_lo, const float* a_scale, float* out, hipStream_t s)
{
    static_assert(GM_ROWS_GU == 128 && GM_ROWS_DN == 256 && GD_ROWS == 256, "the tiles of unit_lists");
    if (d.group != 64 || d.I % 64 || d.D % 64 || P == 0 || !lists.units) return hipErrorInvalidValue;
    const uint32_t n_dim = GATE_UP ? d.I : d.D, k_dim = GATE_UP ? d.D : d.I, div = GATE_UP ? d.K : 1u;
    const uint4* units = lists.units + (GATE_UP ? 0u : lists.slots[0]);
    const uint32_t nt = lists.tiles[GATE_UP ? 0 : 1];
    const dim3 grid(lists.slots[GATE_UP ? 0 : 1] * nt);
    if (reg_supported(L, k_dim) && !lds_weights(P, d.E, nt))
        launch_kernel(k_grouped_reg<GATE_UP>, grid, dim3(GD_WAVES * WAVE), s, d, L, units, sorted_pairs, a_hi, a_lo,
                      a_scale, div, out, n_dim, k_dim, nt);
    else
        launch_kernel(k_grouped_mm<GATE_UP>, grid, dim3(GM_WAVES * WAVE), s, d, L, units, sorted_pairs, a_hi, a_lo,
                      a_scale, div, out, n_dim, k_dim, nt);
    return hipGetLastError();
}

hipError_t launch_grouped_gate_up(const MoeDims& d, const LayerDesc& L, uint32_t P, const UnitLists& lists,
                                  const uint32_t* sorted_pairs, const uint16_t* x_hi,
                                  const uint16_t* x_lo, const float* x_scale, float* h, hipStream_t s)
{
    return launch_grouped<true>(d, L, P, lists, sorted_pairs, x_hi, x_lo, x_scale, h, s);
}

hipError_t launch_grouped_down(const MoeDims& d, const LayerDesc& L, uint32_t P, const UnitLists& lists,
                               const uint32_t* sorted_pairs, const uint16_t* h_hi,
                               const uint16_t* h_lo, const float* h_scale, float* y, hipStream_t s)
{
    return launch_grouped<false>(d, L, P, lists, sorted_pairs, h_hi, h_lo, h_scale, y, s);
}

hipError_t launch_combine_pairs(const float* y, const float* w, uint32_t T, uint32_t K, uint32_t D, float* hidden,
                                hipStream_t s)
{
    if (D % 4) return hipErrorInvalidValue;
    launch_kernel(k_combine_pairs, dim3((D / 4 + 255) / 256, T), dim3(256), s, y, w, K, D, hidden);
    return hipGetLastError();
}

}  // namespace smoe
