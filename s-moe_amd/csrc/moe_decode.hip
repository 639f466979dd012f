// moe_decode.hip -- batch-1 decode MoE block on gfx950.
//
// Two launches per layer; the kernel boundary between them is the layer's
// second global synchronisation point (a launch is cheaper on MI355X than an
// in-kernel grid barrier):
//   k_moe_up       RMSNorm (common.hpp:245-256) + bf16 router GEMV
//                  (common.hpp:293-306) in the first blocks, published as
//                  flag-carrying 64-bit words that every block polls; softmax +
//                  top-k (scout.cpp:77-123) with the renormalisation
//                  (decode.cpp:296-302) block-wide in every block; then the
//                  gate+up+SiLU GEMV of every selected expert in one launch
//                  (kernels.metal:240-337): one wave per block of rows, each
//                  lane owning a fixed 16-byte column chunk of every row, so
//                  its 32 activations stay in VGPRs and the dequant folds into
//                  a per-chunk affine epilogue (kernels.metal:140-145).
//   k_down_combine down GEMV of all k experts (kernels.metal:340-365) with the
//                  routing-weighted combine and the residual add fused
//                  (decode.cpp:482-509): lane p owns (expert, column chunk)
//                  pair p, so every down row of all k experts is one 64-lane
//                  reduction and no per-expert output ever reaches HBM.
//
// Loads of packed nibbles are 128-bit and non-temporal; activations and h
// planes are tiny and stay in L2.
#include <algorithm>
#include <type_traits>

#include "device_common.hpp"
#include "kernels.hpp"
#include "topk.hpp"

namespace smoe {

DispatchTimer& dispatch_timer()
{
    static thread_local DispatchTimer t;
    return t;
}

// ---------------------------------------------------------------------------
// k_topk: Scout::compute_top_k (scout.cpp:718-720) on rows of scores, one
// wave per row, through the same selection k_moe_up uses.
// ---------------------------------------------------------------------------
template <int VPL>
__global__ __launch_bounds__(WAVE)
void k_topk(const float* __restrict__ scores, uint32_t n, uint32_t k, uint32_t norm, uint32_t* __restrict__ ids,
            float* __restrict__ w)
{
    __shared__ uint2 slots[TOPK_SLOTS];
    const size_t row = blockIdx.x;
    float v[VPL];
    topk_load<VPL>(scores + row * n, n, v);
    uint32_t my_id;
    float my_w;
    const uint32_t count = topk_latency<VPL>(v, n, k, norm, my_id, my_w, slots);
    if (threadIdx.x < count) {
        ids[row * k + threadIdx.x] = my_id;
        w[row * k + threadIdx.x] = my_w;
    }
}

// ---------------------------------------------------------------------------
// k_moe_up: RMSNorm + router + softmax/top-k + gate/up/SiLU for one layer.
// One wave per block; grid (at most I / 8, K, T).  Lane l owns the 32 columns of
// chunk l (+64 j) of the hidden dimension throughout.  Every wave:
//   1. loads its hidden and norm-weight chunks and its router rows,
//   2. RMS-normalises them, normed = (x * inv) * w (common.hpp:245-256),
//   3. turns the normed chunk into 4-bit digit words (Q4Act),
//   4. computes its router rows' logits, router_w[row] . normed
//      (common.hpp:293-306), published as flag-carrying 64-bit words,
//   5. polls the E logits of its token and selects the experts itself
//      (softmax + top-k, scout.cpp:77-123; renormalised, decode.cpp:296-302),
//   6. streams its blocks of 8 rows of gate and up of the expert of rank
//      blockIdx.y and writes h = silu(gate) * up (kernels.metal:240-337).
// The logit exchange is XCD-local when the token's block count is a multiple
// of 8: the dispatcher deals consecutive blocks round-robin over the 8 XCDs
// (from some starting XCD), so block b is the (b/8)-th of its XCD, and the
// blocks of every XCD compute all E rows among themselves (rows b/8,
// b/8 + nb/8, ...).  The words then stay in that XCD's L2 (plain stores; the
// pollers' loads are agent-scope) in the copy of its XCC_ID.  Otherwise block
// b < E computes rows b, b + nb, ... and writes every copy through.  A bounded
// spin reports a timeout (err) instead of hanging.  Block 0 of each token
// publishes ids, weights and the expert table.  Steps 1-3 overlap the router
// rows' latency.
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint64_t ll_word(float v) { return (1ull << 32) | __float_as_uint(v); }

constexpr uint32_t SPIN_LIMIT = 1u << 22;
constexpr int UP_RB = 8;   // rows per wave
constexpr int SMOE_G = 64; // SMOE-Q4 group size (shatter_moe.py Q2_GROUP_SIZE)

template <int CPL, int VPL, bool LOCAL, bool LOOP>
__device__ __forceinline__ void moe_up_body(const MoeDims& d, const LayerDesc& L, const float* __restrict__ hv,
                                            uint64_t* __restrict__ ll, float* __restrict__ h,
                                            uint32_t* __restrict__ ids_out, float* __restrict__ w_out,
                                            ExpertPtrs* __restrict__ tbl_out, uint32_t* __restrict__ err)
{
    constexpr int RB = UP_RB;
    const int lane = threadIdx.x;
    const uint32_t tok = blockIdx.z, r = blockIdx.y;
    const uint32_t D = d.D, nch = D >> 5;
    const uint32_t nb = gridDim.x * gridDim.y;
    const uint32_t b = blockIdx.y * gridDim.x + blockIdx.x;
    uint32_t row0, rstep, copy;
    if constexpr (LOCAL) {
        uint32_t xcc;
        asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID, 0, 4)" : "=s"(xcc));
        row0 = b >> 3;
        rstep = nb >> 3;
        copy = xcc & (LL_COPIES - 1);
    } else {
        row0 = b;
        rstep = nb;
        copy = b % LL_COPIES;
    }
    const bool producer = row0 < d.E;
    const bool second = row0 + rstep < d.E;

    // 1. chunk loads (router last, so the norm can start before it lands)
    float4 x[CPL][8];
    uint4 g[CPL][4], rw[CPL][4], rw2[CPL][4];
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
        const uint32_t c = min(lane + WAVE * j, nch - 1);
#pragma unroll
        for (int q = 0; q < 8; ++q) x[j][q] = load_f4(hv + c * 32 + q * 4);
#pragma unroll
        for (int q = 0; q < 4; ++q) g[j][q] = load_u4(L.norm_w + c * 32 + q * 8);
    }
    // router rows: plain loads (the previous layer's down kernel may have
    // left them in this XCD's L2)
    if (producer) {
        const uint16_t* wr = L.router_w + static_cast<size_t>(row0) * D;
#pragma unroll
        for (int j = 0; j < CPL; ++j) {
            const uint32_t c = min(lane + WAVE * j, nch - 1);
#pragma unroll
            for (int q = 0; q < 4; ++q) rw[j][q] = load_u4(wr + c * 32 + q * 8);
        }
        if (second) {
            const uint16_t* wr2 = L.router_w + static_cast<size_t>(row0 + rstep) * D;
#pragma unroll
            for (int j = 0; j < CPL; ++j) {
                const uint32_t c = min(lane + WAVE * j, nch - 1);
#pragma unroll
                for (int q = 0; q < 4; ++q) rw2[j][q] = load_u4(wr2 + c * 32 + q * 8);
            }
        }
    }
    // 2. RMS norm over the wave's D columns
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
    // rms_norm_bf16 (common.hpp:245-256): inv = 1 / sqrt(ss / n + 1e-6)
    const float inv = 1.0f / sqrtf(ss / static_cast<float>(D) + 1e-6f);
    float a[CPL][32];
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const uint32_t g0 = (q & 1) ? g[j][q >> 1].z : g[j][q >> 1].x;
            const uint32_t g1 = (q & 1) ? g[j][q >> 1].w : g[j][q >> 1].y;
            a[j][4 * q + 0] = (x[j][q].x * inv) * bf16_to_f32(g0 & 0xFFFFu);
            a[j][4 * q + 1] = (x[j][q].y * inv) * bf16_to_f32(g0 >> 16);
            a[j][4 * q + 2] = (x[j][q].z * inv) * bf16_to_f32(g1 & 0xFFFFu);
            a[j][4 * q + 3] = (x[j][q].w * inv) * bf16_to_f32(g1 >> 16);
        }
    }
    // 4. router rows row0, row0 + rstep, ... (padding lanes hold normed 0)
    uint64_t* llc = ll + copy * ll_copy_words(d.E);
    auto publish = [&](uint32_t row, float acc) {
        if constexpr (LOCAL) {
            if (lane == 0)
                __hip_atomic_store(llc + row, ll_word(acc), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
        } else {
            if (lane < static_cast<int>(LL_COPIES))
                __hip_atomic_store(ll + lane * ll_copy_words(d.E) + row, ll_word(acc), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        }
    };
    auto row_dot = [&](const uint4 (&w)[CPL][4]) {
        float acc = 0.f;
#pragma unroll
        for (int j = 0; j < CPL; ++j) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t w4[4] = {w[j][q].x, w[j][q].y, w[j][q].z, w[j][q].w};
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    acc = fmaf(bf16_to_f32(w4[t] & 0xFFFFu), a[j][8 * q + 2 * t], acc);
                    acc = fmaf(bf16_to_f32(w4[t] >> 16), a[j][8 * q + 2 * t + 1], acc);
                }
            }
        }
        return wave_sum(acc);
    };
    if (producer) {
        publish(row0, row_dot(rw));
        if (second) {
            publish(row0 + rstep, row_dot(rw2));
            for (uint32_t row = row0 + 2 * rstep; row < d.E; row += rstep) {
                const uint16_t* wr = L.router_w + static_cast<size_t>(row) * D;
#pragma unroll
                for (int j = 0; j < CPL; ++j) {
                    const uint32_t c = min(lane + WAVE * j, nch - 1);
#pragma unroll
                    for (int q = 0; q < 4; ++q) rw[j][q] = load_u4(wr + c * 32 + q * 8);
                }
                publish(row, row_dot(rw));
            }
        }
    }
    // 3. digit form of the normed chunk (overlaps the logit exchange)
    Q4Act qa[CPL];
#pragma unroll
    for (int j = 0; j < CPL; ++j) q4_act_from_floats(a[j], qa[j]);
    // 5. wait for the E logits (in this block's copy), then select
    float v[VPL];
    {
        uint32_t spins = 0;
        bool all;
        do {
            all = true;
            // every load issued before any is waited on (padding lanes re-read word E-1)
#pragma unroll
            for (int j = 0; j < VPL; ++j) {
                const uint32_t pos = lane + WAVE * j;
                const uint64_t w64 =
                    __hip_atomic_load(llc + min(pos, d.E - 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                v[j] = __uint_as_float(static_cast<uint32_t>(w64));
                all &= pos >= d.E || (w64 >> 32) != 0;
            }
            all = __ballot(!all) == 0;
            if (!all && ++spins > SPIN_LIMIT) {
                if (lane == 0) atomicOr(err, 1u);
                break;
            }
        } while (!all);
    }
    uint32_t my_id;
    float my_w;
    __shared__ uint2 slots[TOPK_SLOTS];
    topk_latency<VPL>(v, d.E, d.K, d.norm_topk, my_id, my_w, slots);
    const uint32_t expert = readlane_u32(my_id, r);

    if (b == 0 && static_cast<uint32_t>(lane) < d.K) {
        const size_t o = static_cast<size_t>(tok) * d.K + lane;
        ids_out[o] = my_id;
        w_out[o] = my_w;
        const uint8_t* bb = L.experts + static_cast<size_t>(my_id) * L.stride;
        ExpertPtrs e;
        e.pg = bb + L.off[0];
        e.sg = reinterpret_cast<const uint16_t*>(bb + L.off[1]);
        e.pu = bb + L.off[2];
        e.su = reinterpret_cast<const uint16_t*>(bb + L.off[3]);
        e.pd = bb + L.off[4];
        e.sd = reinterpret_cast<const uint16_t*>(bb + L.off[5]);
        e.slot = lane;
        e.pad_ = 0;
        tbl_out[o] = e;
    }

    // 6. row block blockIdx.x of 8 rows of gate and up, and with LOOP + gridDim.x,
    // ...: every weight load of a block in flight before any is used, and with one
    // chunk a lane the next block's as well
    const uint8_t* blob = L.experts + static_cast<size_t>(expert) * L.stride;
    const uint8_t* pa = blob + L.off[0];
    const uint16_t* sa = reinterpret_cast<const uint16_t*>(blob + L.off[1]);
    const uint8_t* pb = blob + L.off[2];
    const uint16_t* sb = reinterpret_cast<const uint16_t*>(blob + L.off[3]);
    const uint32_t row_bytes = D >> 1, row_scales = D / SMOE_G;
    float* o = h + (static_cast<size_t>(tok) * d.K + r) * d.I;
    struct Rows {
        uint4 va[RB][CPL], vb[RB][CPL];
        uint16_t sva[RB][CPL], svb[RB][CPL];
    };
    auto load_rows = [&](uint32_t rb, Rows& w) {
#pragma unroll
        for (int i = 0; i < RB; ++i) {
            const size_t row = rb * RB + i;
#pragma unroll
            for (int j = 0; j < CPL; ++j) {
                const uint32_t c = min(lane + WAVE * j, nch - 1);
                w.va[i][j] = load_stream_u4(pa + row * row_bytes + c * 16);
                w.vb[i][j] = load_stream_u4(pb + row * row_bytes + c * 16);
                w.sva[i][j] = load_stream_u16(sa + row * row_scales + (c * 32) / SMOE_G);
                w.svb[i][j] = load_stream_u16(sb + row * row_scales + (c * 32) / SMOE_G);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto do_rows = [&](uint32_t rb, const Rows& w) {
        // per-lane partial dots: value 2i = gate row i, 2i + 1 = up row i
        float part[2 * RB];
#pragma unroll
        for (int i = 0; i < RB; ++i) {
            float ga = 0.f, ua = 0.f;
#pragma unroll
            for (int j = 0; j < CPL; ++j) {
                ga = fmaf(f16_bits_to_f32(w.sva[i][j]), q4_chunk_dot8(w.va[i][j], qa[j]), ga);
                ua = fmaf(f16_bits_to_f32(w.svb[i][j]), q4_chunk_dot8(w.vb[i][j], qa[j]), ua);
            }
            part[2 * i] = ga;
            part[2 * i + 1] = ua;
        }
        // lane l holds the total of value l >> SH
        constexpr int SH = 6 - ilog2(2 * RB);
        const float tot = wave_sum_rows<2 * RB>(part);
        const float gv = __shfl(tot, (2 * lane) << SH);
        const float uv = __shfl(tot, (2 * lane + 1) << SH);
        // silu(z) = z * (1 / (1 + exp(-z)))  (kernels.metal:61-63, :334-336), all rows at once
        if (lane < RB) o[rb * RB + lane] = (gv * (1.0f / (1.0f + expf(-gv)))) * uv;
    };
    const uint32_t nrb = d.I / RB, step = gridDim.x;
    Rows wa;
    if constexpr (!LOOP) {
        load_rows(blockIdx.x, wa);
        do_rows(blockIdx.x, wa);
    } else if constexpr (CPL == 1) {
        Rows wb;
        load_rows(blockIdx.x, wa);
        for (uint32_t rb = blockIdx.x; rb < nrb; rb += 2 * step) {
            if (rb + step < nrb) load_rows(rb + step, wb);
            do_rows(rb, wa);
            if (rb + step >= nrb) break;
            if (rb + 2 * step < nrb) load_rows(rb + 2 * step, wa);
            do_rows(rb + step, wb);
        }
    } else {
        for (uint32_t rb = blockIdx.x; rb < nrb; rb += step) {
            load_rows(rb, wa);
            do_rows(rb, wa);
        }
    }
}

template <int CPL, int VPL, bool LOCAL, bool LOOP>
__global__ __launch_bounds__(WAVE)
void k_moe_up(MoeDims d, LayerDesc L, const float* __restrict__ hidden, uint64_t* __restrict__ ll_all,
              float* __restrict__ h, uint32_t* __restrict__ ids_out, float* __restrict__ w_out,
              ExpertPtrs* __restrict__ tbl_out, uint32_t* __restrict__ err)
{
    const uint32_t tok = blockIdx.z;
    const float* hv = hidden + static_cast<size_t>(tok) * d.D;
    uint64_t* ll = ll_all + static_cast<size_t>(tok) * ll_token_words(d.E);
    moe_up_body<CPL, VPL, LOCAL, LOOP>(d, L, hv, ll, h, ids_out, w_out, tbl_out, err);
}

// ---------------------------------------------------------------------------
// k_q4_rows: rows of SMOE-Q4 matrices dotted with activation vectors, one
// token per blockIdx.y (reference surface).
//   GATE_UP: rows = I of gate and up, cols = D, x = normed token,
//            out = silu(gate.x) * (up.x)
//   DOWN:    rows = D of down, cols = I, x = h of the table entry's slot
// One wave = RB consecutive rows of one table entry; lane owns chunks
// c = lane + 64 j of every row (CPL chunks), 32 activations each in VGPRs.
// ---------------------------------------------------------------------------
template <int CPL, int RB, bool GATE_UP>
__global__ __launch_bounds__(256)
void k_q4_rows(MoeDims d, ExpertTable tbl, uint32_t n_exp, const float* __restrict__ x, uint32_t x_slot_stride,
               uint32_t x_tok_stride, float* __restrict__ out, uint32_t out_stride, uint32_t out_tok_stride)
{
    const int lane = threadIdx.x & 63;
    const uint32_t wave_id = blockIdx.x * 4 + (threadIdx.x >> 6);
    const uint32_t rows = GATE_UP ? d.I : d.D;
    const uint32_t cols = GATE_UP ? d.D : d.I;
    const uint32_t nrb = rows / RB;
    if (wave_id >= n_exp * nrb) return;
    const uint32_t r = wave_id / nrb;
    const uint32_t row0 = (wave_id - r * nrb) * RB;
    const ExpertPtrs& e = tbl.e[r];
    const uint32_t tok = blockIdx.y;
    const float* xv = x + static_cast<size_t>(tok) * x_tok_stride +
                      (GATE_UP ? 0 : static_cast<size_t>(e.slot) * x_slot_stride);
    const uint32_t nch = cols >> 5;
    const uint32_t row_bytes = cols >> 1;
    const uint32_t row_scales = cols / d.group;

    const uint8_t* pa = GATE_UP ? e.pg : e.pd;
    const uint16_t* sa = GATE_UP ? e.sg : e.sd;
    const uint8_t* pb = e.pu;
    const uint16_t* sb = e.su;

    float xr[CPL][32];
    float xsum[CPL];
    uint4 va[RB][CPL], vb[RB][CPL];
    uint16_t sva[RB][CPL], svb[RB][CPL];
#pragma unroll
    for (int i = 0; i < RB; ++i) {
        const size_t row = row0 + i;
#pragma unroll
        for (int j = 0; j < CPL; ++j) {
            const uint32_t c = min(lane + WAVE * j, nch - 1);
            va[i][j] = load_stream_u4(pa + row * row_bytes + c * 16);
            sva[i][j] = load_stream_u16(sa + row * row_scales + (c * 32) / d.group);
            if (GATE_UP) {
                vb[i][j] = load_stream_u4(pb + row * row_bytes + c * 16);
                svb[i][j] = load_stream_u16(sb + row * row_scales + (c * 32) / d.group);
            }
        }
    }
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
        const uint32_t c = min(lane + WAVE * j, nch - 1);
        const bool ok = lane + WAVE * j < nch;
        xsum[j] = 0.f;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const float4 v = load_f4(xv + c * 32 + q * 4);
            xr[j][q * 4 + 0] = ok ? v.x : 0.f;
            xr[j][q * 4 + 1] = ok ? v.y : 0.f;
            xr[j][q * 4 + 2] = ok ? v.z : 0.f;
            xr[j][q * 4 + 3] = ok ? v.w : 0.f;
        }
#pragma unroll
        for (int q = 0; q < 32; ++q) xsum[j] += xr[j][q];
    }
    float* o = out + static_cast<size_t>(tok) * out_tok_stride + static_cast<size_t>(e.slot) * out_stride;
    static_assert(RB == 4, "four rows a store");
    float y[RB];
#pragma unroll
    for (int i = 0; i < RB; ++i) {
        float aa = 0.f, ab = 0.f;
#pragma unroll
        for (int j = 0; j < CPL; ++j) {
            aa += q4_chunk_epilogue(f16_bits_to_f32(sva[i][j]), q4_chunk_dot(va[i][j], xr[j]), xsum[j]);
            if (GATE_UP)
                ab += q4_chunk_epilogue(f16_bits_to_f32(svb[i][j]), q4_chunk_dot(vb[i][j], xr[j]), xsum[j]);
        }
        aa = wave_sum(aa);
        if (GATE_UP) ab = wave_sum(ab);
        // silu(z) = z * (1 / (1 + exp(-z)))  (kernels.metal:61-63, :334-336)
        y[i] = GATE_UP ? (aa * (1.0f / (1.0f + expf(-aa)))) * ab : aa;
    }
    // one store a wave: `out` of the down rows is host memory
    if (lane == 0) *reinterpret_cast<float4*>(o + row0) = make_float4(y[0], y[1], y[2], y[3]);
}

// ---------------------------------------------------------------------------
// k_ffn_tokens: one expert's rows times several token vectors (reference
// surface, smoe_metal_fused_ffn_batch), on v_mfma_f32_16x16x4_f32 (fp32
// products and sums).
//   GATE_UP: rows = I, cols = D, out[t][row] = silu(gate.x) * (up.x)
//   DOWN:    rows = D, cols = I, out[t][row] = down.h
// Block: 16 tokens x two 16-row subtiles (16 rows of gate and of up, or 32 of
// down); its NW waves share the columns, KB at a time (KB = 64, or 32 for
// groups of 32), and their partial tiles are added through LDS.  A lane (m16, q)
// of a KB-column step holds columns KB / 4 q .. of token m16 (A) and of row m16
// (B): MFMA step j takes the lane's j-th, so K index q stands for column KB / 4 q + j
// on both sides and every load is contiguous.  Weights enter as c - 7.5
// (exact); s / 7.5 scales each step's sums.  The MFMA work of a whole call is
// under 4 us, so the tiles are small to spread one expert over the chip.  37
// tokens of a 30B expert: 12.4 us (gate/up) + 6.4 us (down), against 19.5 + 20.2
// for a wave per four rows and token (k_q4_rows), which converts the codes again for
// every token; the relative error against fp64 falls from 7e-7 to 3e-7.
// ---------------------------------------------------------------------------
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr uint32_t FFN_FEW_TOKENS = 8;   // up to here k_q4_rows (launch_tokens)

template <bool GATE_UP, int KB, int NW>
__global__ __launch_bounds__(NW * WAVE)
void k_ffn_tokens(MoeDims d, ExpertPtrs e, const float* __restrict__ x, float* __restrict__ out, uint32_t n_tok)
{
    constexpr int U = 4;                         // steps in flight
    constexpr int KL = KB / 4;                   // columns of a lane in a step
    __shared__ float s_acc[NW][2][16][17];
    const int lane = threadIdx.x & 63, m16 = lane & 15, q = lane >> 4;
    const uint32_t wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t rows = GATE_UP ? d.I : d.D, cols = GATE_UP ? d.D : d.I;
    const uint32_t nb = cols / KB, row_bytes = cols >> 1, row_scales = cols / d.group;
    const uint32_t row0 = blockIdx.x * (GATE_UP ? 16 : 32), t0 = blockIdx.y * 16;
    const uint8_t* pw[2];
    const uint16_t* ps[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const size_t row = row0 + (GATE_UP ? 0 : 16 * j) + m16;
        pw[j] = (GATE_UP ? (j ? e.pu : e.pg) : e.pd) + row * row_bytes + q * (KL / 2);
        ps[j] = (GATE_UP ? (j ? e.su : e.sg) : e.sd) + row * row_scales;
    }
    const float* px = x + static_cast<size_t>(min(t0 + m16, n_tok - 1)) * cols + q * KL;

    f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    for (uint32_t b0 = wv; b0 < nb; b0 += NW * U) {
        uint32_t w[U][2][KL / 8];
        uint16_t sv[U][2];
        float4 xv[U][KL / 4];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t b = min(b0 + u * NW, nb - 1);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const uint32_t* p = reinterpret_cast<const uint32_t*>(pw[j] + b * (KB / 2));
#pragma unroll
                for (int k = 0; k < KL / 8; ++k) w[u][j][k] = gptr(p)[k];
                sv[u][j] = *gptr(ps[j] + b * KB / d.group);
            }
#pragma unroll
            for (int k = 0; k < KL / 4; ++k) xv[u][k] = load_f4(px + b * KB + 4 * k);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (b0 + u * NW >= nb) break;
            f32x4 t[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
            for (int k = 0; k < KL / 8; ++k) {
                float wf[2][8];
#pragma unroll
                for (int j = 0; j < 2; ++j) q4_word_floats(w[u][j][k], wf[j]);
                const float4 a = xv[u][2 * k], c = xv[u][2 * k + 1];
                const float xf[8] = {a.x, a.y, a.z, a.w, c.x, c.y, c.z, c.w};
#pragma unroll
                for (int i = 0; i < 8; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        t[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(xf[i], wf[j][i], t[j], 0, 0, 0);
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const float s = f16_bits_to_f32(sv[u][j]) * (1.0f / 7.5f);
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[j][i] = fmaf(s, t[j][i], acc[j][i]);
            }
        }
    }
    // D[4 q + i][m16]: token 4 q + i, row m16 of each subtile
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) s_acc[wv][j][4 * q + i][m16] = acc[j][i];
    __syncthreads();
    for (uint32_t o = threadIdx.x; o < (GATE_UP ? 256u : 512u); o += NW * WAVE) {
        const uint32_t n = o & 15, j = GATE_UP ? 0 : (o >> 4) & 1, t = GATE_UP ? o >> 4 : o >> 5;
        if (t0 + t >= n_tok) continue;
        float v[2] = {0.f, 0.f};
#pragma unroll
        for (int k = 0; k < NW; ++k) {
            v[0] += s_acc[k][j][t][n];
            if (GATE_UP) v[1] += s_acc[k][1][t][n];
        }
        // silu(z) = z * (1 / (1 + exp(-z)))  (kernels.metal:61-63, :334-336)
        const float y = GATE_UP ? (v[0] * (1.0f / (1.0f + expf(-v[0])))) * v[1] : v[0];
        out[static_cast<size_t>(t0 + t) * rows + row0 + 16 * j + n] = y;
    }
}

// ---------------------------------------------------------------------------
// k_down_combine: hidden[row] += sum_r w_r * (down_r[row] . h_r).
// Lane p of the block owns (expert, 32-column chunk) pair p of the k experts'
// down rows (PPL pairs per lane); its 32 h values are turned into digit words
// once and reused for the block's DOWN_RB rows, so each row of all k experts
// is one block-wide reduction: a transposed wave reduction over the rows,
// then the waves' partials through LDS.  Loads go out in dependency order:
// expert table and h first, the down weights as soon as the table lands; the
// h conversion overlaps the weight fetch.
// ---------------------------------------------------------------------------
constexpr int DOWN_RB = 8;
constexpr int DOWN_MAX_WAVES = 8;

template <int PPL, bool LOOP>
__global__ __launch_bounds__(DOWN_MAX_WAVES * WAVE)
void k_down_combine(MoeDims d, const ExpertPtrs* __restrict__ tbl, const float* __restrict__ h,
                    const float* __restrict__ w, float* __restrict__ hidden, uint64_t* __restrict__ ll_all)
{
    constexpr int RB = DOWN_RB;
    // re-arm the routing exchange words of this token for the next k_moe_up
    // (every k_moe_up that read them has finished: this is the next kernel)
    if (blockIdx.x == 0) {
        uint64_t* ll = ll_all + static_cast<size_t>(blockIdx.y) * ll_token_words(d.E);
        for (uint32_t i = threadIdx.x; i < LL_COPIES * d.E; i += blockDim.x)
            ll[(i / d.E) * ll_copy_words(d.E) + i % d.E] = 0;
    }
    __shared__ float part[2][DOWN_MAX_WAVES][RB];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int nw = blockDim.x >> 6;
    const uint32_t tok = blockIdx.y;
    tbl += static_cast<size_t>(tok) * d.K;
    h += static_cast<size_t>(tok) * d.K * d.I;
    w += static_cast<size_t>(tok) * d.K;
    hidden += static_cast<size_t>(tok) * d.D;
    const uint32_t cpr = d.I >> 5;
    const uint32_t npairs = d.K * cpr;
    const uint32_t row_bytes = d.I >> 1, row_scales = d.I / SMOE_G;

    const uint8_t* pd[PPL];
    const uint16_t* sd[PPL];
    uint32_t cc[PPL], rr[PPL];
    bool ok[PPL];
    float4 hx[PPL][8];
    float wr[PPL];
#pragma unroll
    for (int j = 0; j < PPL; ++j) {
        const uint32_t p0 = (wv * PPL + j) * WAVE + lane;
        ok[j] = p0 < npairs;
        const uint32_t p = min(p0, npairs - 1);
        rr[j] = p / cpr;
        cc[j] = p - rr[j] * cpr;
        pd[j] = tbl[rr[j]].pd;
        sd[j] = tbl[rr[j]].sd;
    }
#pragma unroll
    for (int j = 0; j < PPL; ++j) {
        const float* hv = h + static_cast<size_t>(rr[j]) * d.I + cc[j] * 32;
#pragma unroll
        for (int q = 0; q < 8; ++q) hx[j][q] = load_f4(hv + q * 4);
        wr[j] = w[rr[j]];
    }
    __builtin_amdgcn_sched_barrier(0);
    // row block blockIdx.x of RB rows, and with LOOP + gridDim.x, ..., the next
    // block's weights requested before this one's are used
    struct Rows {
        uint4 v[RB][PPL];
        uint16_t sv[RB][PPL];
    };
    auto load_rows = [&](uint32_t rb, Rows& x) {
#pragma unroll
        for (int i = 0; i < RB; ++i) {
            const size_t row = rb * RB + i;
#pragma unroll
            for (int j = 0; j < PPL; ++j) {
                x.v[i][j] = load_stream_u4(pd[j] + row * row_bytes + cc[j] * 16);
                x.sv[i][j] = load_stream_u16(sd[j] + row * row_scales + (cc[j] * 32) / SMOE_G);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    const uint32_t nrb = d.D / RB, step = gridDim.x;
    Rows xa;
    load_rows(blockIdx.x, xa);
    Q4Act qh[PPL];
#pragma unroll
    for (int j = 0; j < PPL; ++j) {
        float a[32];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            a[q * 4 + 0] = hx[j][q].x;
            a[q * 4 + 1] = hx[j][q].y;
            a[q * 4 + 2] = hx[j][q].z;
            a[q * 4 + 3] = hx[j][q].w;
        }
        q4_act_from_floats(a, qh[j]);
        if (!ok[j]) wr[j] = 0.f;   // pairs past the end contribute nothing
    }
    auto do_rows = [&](uint32_t rb, const Rows& x, int buf) {
        float acc[RB];
#pragma unroll
        for (int i = 0; i < RB; ++i) {
            acc[i] = 0.f;
#pragma unroll
            for (int j = 0; j < PPL; ++j) {
                const float y = f16_bits_to_f32(x.sv[i][j]) * q4_chunk_dot8(x.v[i][j], qh[j]);
                acc[i] = fmaf(wr[j], y, acc[i]);
            }
        }
        // lane l holds the wave's total of row l >> SH
        constexpr int SH = 6 - ilog2(RB);
        const float tot = wave_sum_rows<RB>(acc);
        if ((lane & ((1 << SH) - 1)) == 0) part[buf][wv][lane >> SH] = tot;
        // (two buffers: the next block's partials go to the other one, and the
        // one after that is past the barrier that every reader has reached)
        __syncthreads();
        if (threadIdx.x < RB) {
            float t = 0.f;
            for (int q = 0; q < nw; ++q) t += part[buf][q][threadIdx.x];
            const uint32_t row = rb * RB + threadIdx.x;
            hidden[row] = hidden[row] + t;
        }
    };
    if constexpr (LOOP) {
        Rows xb;
        for (uint32_t rb = blockIdx.x; rb < nrb; rb += 2 * step) {
            if (rb + step < nrb) load_rows(rb + step, xb);
            do_rows(rb, xa, 0);
            if (rb + step >= nrb) break;
            if (rb + 2 * step < nrb) load_rows(rb + 2 * step, xa);
            do_rows(rb + step, xb, 1);
        }
    } else {
        do_rows(blockIdx.x, xa, 0);
    }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
template <int CPL, int VPL>
static void moe_up_v(dim3 grid, bool loop, hipStream_t s, const MoeDims& d, const LayerDesc& L, const float* hidden,
                     uint64_t* ll, float* h, uint32_t* ids, float* w, ExpertPtrs* tbl, uint32_t* err)
{
    // XCD-local logit exchange when every XCD receives the same number of
    // blocks of each token, they cover the router rows in at most two each,
    // and the whole grid is resident at once (the dispatcher's round-robin
    // over the XCDs is then unbroken)
    const uint32_t nb = grid.x * grid.y;
    const bool local = nb % 8 == 0 && nb / 8 * 2 >= d.E && nb * grid.z <= 1024;
    auto go = [&](auto* k) { launch_kernel(k, grid, dim3(WAVE), s, d, L, hidden, ll, h, ids, w, tbl, err); };
    if (local) loop ? go(k_moe_up<CPL, VPL, true, true>) : go(k_moe_up<CPL, VPL, true, false>);
    else loop ? go(k_moe_up<CPL, VPL, false, true>) : go(k_moe_up<CPL, VPL, false, false>);
}

template <int CPL>
static void moe_up_c(dim3 grid, bool loop, hipStream_t s, const MoeDims& d, const LayerDesc& L, const float* hidden,
                     uint64_t* ll, float* h, uint32_t* ids, float* w, ExpertPtrs* tbl, uint32_t* err)
{
    if (d.E <= 128)
        moe_up_v<CPL, 2>(grid, loop, s, d, L, hidden, ll, h, ids, w, tbl, err);
    else
        moe_up_v<CPL, 8>(grid, loop, s, d, L, hidden, ll, h, ids, w, tbl, err);
}

hipError_t launch_moe_up(const MoeDims& d, const LayerDesc& L, const float* hidden, uint32_t n_tok, uint64_t* ll,
                         float* h, uint32_t* ids, float* w, ExpertPtrs* tbl, uint32_t* err, hipStream_t s)
{
    if (d.group != 64 || d.E > SMOE_TOPK_MAX_N || d.I % UP_RB) return hipErrorInvalidValue;
    const uint32_t row_blocks = d.I / UP_RB;
    // Several row blocks a wave once the waves outnumber what the chip holds at
    // two a SIMD (2048; one a SIMD with four chunks a lane, D > 4096, where such a
    // grid takes two rounds): the norm, the digits and the top-k, half of a wave's
    // VALU work with one block, are then done once per wave (11 tokens of the
    // 30B shape 52 -> 33 us, 24 tokens 107 -> 60; with waves for one or three a
    // SIMD 40 and 36).  Grids between one and two a SIMD fold to one (2 tokens 14.0
    // -> 12.7: every wave then has its SIMD to itself; the logit exchange stays as
    // it was, 48 waves an XCD being too few for 128 rows).
    const uint32_t waves = row_blocks * d.K * n_tok;
    const uint32_t most = std::max(1u, (n_tok > 1 && waves > 1024 && waves <= 2048 ? 1024u : 2048u) / (d.K * n_tok));
    const uint32_t iters = (row_blocks + most - 1) / most;
    const dim3 grid((row_blocks + iters - 1) / iters, d.K, n_tok);
    const uint32_t cpl = (d.D / 32 + WAVE - 1) / WAVE;   // 32-column chunks per lane
    if (cpl == 1) moe_up_c<1>(grid, iters > 1, s, d, L, hidden, ll, h, ids, w, tbl, err);
    else if (cpl == 2) moe_up_c<2>(grid, iters > 1, s, d, L, hidden, ll, h, ids, w, tbl, err);
    else if (cpl <= 4) moe_up_c<4>(grid, iters > 1, s, d, L, hidden, ll, h, ids, w, tbl, err);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t launch_topk(const float* scores, uint32_t rows, uint32_t n, uint32_t k,
                       uint32_t norm, uint32_t* ids, float* w, hipStream_t s)
{
    if (topk_vpl(n) == 2)
        launch_kernel(k_topk<2>, dim3(rows), dim3(WAVE), s, scores, n, k, norm, ids, w);
    else
        launch_kernel(k_topk<8>, dim3(rows), dim3(WAVE), s, scores, n, k, norm, ids, w);
    return hipGetLastError();
}

template <bool GATE_UP>
static hipError_t launch_rows(const MoeDims& d, const ExpertTable& tbl, uint32_t n_exp, const float* x,
                              uint32_t x_slot_stride, uint32_t x_tok_stride, float* out, uint32_t out_stride,
                              uint32_t out_tok_stride, uint32_t n_tok, hipStream_t s)
{
    constexpr int RB = 4;
    const uint32_t rows = GATE_UP ? d.I : d.D;
    const uint32_t cols = GATE_UP ? d.D : d.I;
    const uint32_t nch = cols / 32;
    const uint32_t cpl = (nch + WAVE - 1) / WAVE;
    const uint32_t waves = n_exp * (rows / RB);
    if (n_exp == 0 || n_exp > ExpertTable::MAX) return hipErrorInvalidValue;
    const dim3 grid((waves + 3) / 4, n_tok);
#define SMOE_ROWS_CASE(C)                                                                                      \
    case C:                                                                                                    \
        launch_kernel(k_q4_rows<C, RB, GATE_UP>, grid, dim3(256), s, d, tbl, n_exp, x, x_slot_stride,          \
                      x_tok_stride, out, out_stride, out_tok_stride);                                          \
        break;
    switch (cpl) {
        SMOE_ROWS_CASE(1)
        SMOE_ROWS_CASE(2)
        SMOE_ROWS_CASE(3)
        SMOE_ROWS_CASE(4)
        default: return hipErrorInvalidValue;
    }
#undef SMOE_ROWS_CASE
    return hipGetLastError();
}

hipError_t launch_gate_up(const MoeDims& d, const ExpertTable& tbl, uint32_t n_exp, const float* x, float* h,
                          uint32_t h_stride, hipStream_t s)
{
    return launch_rows<true>(d, tbl, n_exp, x, 0, 0, h, h_stride, 0, 1, s);
}

hipError_t launch_down_slots(const MoeDims& d, const ExpertTable& tbl, uint32_t n_exp, const float* h,
                             uint32_t h_stride, float* out, uint32_t out_stride, hipStream_t s)
{
    return launch_rows<false>(d, tbl, n_exp, h, h_stride, 0, out, out_stride, 0, 1, s);
}

template <bool GATE_UP>
static hipError_t launch_tokens(const MoeDims& d, const ExpertPtrs& e, const float* x, float* out, uint32_t n_tok,
                                hipStream_t s)
{
    const uint32_t rows = GATE_UP ? d.I : d.D, cols = GATE_UP ? d.D : d.I;
    if (n_tok == 0 || rows == 0 || cols == 0 || rows % 32 || cols % d.group || d.group % 32) return hipErrorInvalidValue;
    // Few tokens: a wave per four rows and token (5 tokens of a 30B expert 13.2
    // us against 17.0 for the MFMA tiles, whose 48 blocks leave most CUs idle;
    // 16 tokens 22.3 against 18.6).  The table's slot 0 and the token strides
    // address plain matrices.
    if (n_tok <= FFN_FEW_TOKENS) {
        ExpertTable tbl{};
        tbl.e[0] = e;
        return launch_rows<GATE_UP>(d, tbl, 1, x, 0, cols, out, 0, rows, n_tok, s);
    }
    const dim3 grid(rows / (GATE_UP ? 16 : 32), (n_tok + 15) / 16);
    // eight waves share the columns of a long row (three or more steps each)
    const uint32_t kb = d.group % 64 ? 32 : 64;
    const bool w8 = cols / kb >= 24;
    if (kb == 64 && w8) launch_kernel(k_ffn_tokens<GATE_UP, 64, 8>, grid, dim3(512), s, d, e, x, out, n_tok);
    else if (kb == 64) launch_kernel(k_ffn_tokens<GATE_UP, 64, 4>, grid, dim3(256), s, d, e, x, out, n_tok);
    else if (w8) launch_kernel(k_ffn_tokens<GATE_UP, 32, 8>, grid, dim3(512), s, d, e, x, out, n_tok);
    else launch_kernel(k_ffn_tokens<GATE_UP, 32, 4>, grid, dim3(256), s, d, e, x, out, n_tok);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// k_stage_in: n4 float4 from pinned host memory to the device, in stream order
// ahead of the kernels that read them.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256)
void k_stage_in(const float4* __restrict__ src, float4* __restrict__ dst, uint32_t n4)
{
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < n4) dst[i] = src[i];
}

hipError_t launch_stage_in(const float* src, float* dst, uint32_t n, hipStream_t s)
{
    if (n == 0 || n % 4) return hipErrorInvalidValue;
    launch_kernel(k_stage_in, dim3((n / 4 + 255) / 256), dim3(256), s, reinterpret_cast<const float4*>(src),
                  reinterpret_cast<float4*>(dst), n / 4);
    return hipGetLastError();
}

hipError_t launch_gate_up_tokens(const MoeDims& d, const ExpertPtrs& e, const float* x, float* h, uint32_t n_tok,
                                 hipStream_t s)
{
    return launch_tokens<true>(d, e, x, h, n_tok, s);
}

hipError_t launch_down_tokens(const MoeDims& d, const ExpertPtrs& e, const float* h, float* out, uint32_t n_tok,
                              hipStream_t s)
{
    return launch_tokens<false>(d, e, h, out, n_tok, s);
}

hipError_t launch_down_combine(const MoeDims& d, const ExpertPtrs* tbl, const float* h, const float* w,
                               float* hidden, uint64_t* ll, uint32_t n_tok, hipStream_t s)
{
    // one (expert, chunk) pair per lane while the block fits in DOWN_MAX_WAVES waves
    const uint32_t npairs = d.K * (d.I / 32);
    uint32_t ppl = 1;
    while (ppl < 4 && (npairs + 64u * ppl - 1) / (64u * ppl) > DOWN_MAX_WAVES) ppl *= 2;
    const uint32_t nw = (npairs + 64u * ppl - 1) / (64u * ppl);
    if (nw > DOWN_MAX_WAVES || d.D % DOWN_RB) return hipErrorInvalidValue;
    // Several row blocks a block, with one pair a lane (the next rows' registers),
    // once the waves outnumber what the chip holds at three a SIMD: h is converted
    // once for all of them (11 tokens of the 30B shape 22.4 -> 20.1 us, of
    // the 235B shape 69.6 -> 63.4; for two a SIMD 22.1 and 84).
    const uint32_t row_blocks = d.D / DOWN_RB;
    const uint32_t most = ppl == 1 ? std::max(1u, 3072u / (nw * n_tok)) : row_blocks;
    const uint32_t iters = (row_blocks + most - 1) / most;
    const dim3 grid((row_blocks + iters - 1) / iters, n_tok), block(nw * WAVE);
    if (ppl == 1 && iters > 1) launch_kernel(k_down_combine<1, true>, grid, block, s, d, tbl, h, w, hidden, ll);
    else if (ppl == 1) launch_kernel(k_down_combine<1, false>, grid, block, s, d, tbl, h, w, hidden, ll);
    else if (ppl == 2) launch_kernel(k_down_combine<2, false>, grid, block, s, d, tbl, h, w, hidden, ll);
    else launch_kernel(k_down_combine<4, false>, grid, block, s, d, tbl, h, w, hidden, ll);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// k_matvec_bf16: out[r] = sum_c bf16(W[r][c]) * x[c] (common.hpp:293-306), one
// wave per row, any cols (the dense-trunk projections of the reference
// surface, metal_bridge.h:157-161; not on the MoE hot path).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256)
void k_matvec_bf16(const uint16_t* __restrict__ W, const float* __restrict__ x, float* __restrict__ out,
                   uint32_t rows, uint32_t cols)
{
    const int lane = threadIdx.x & 63;
    const uint32_t r = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (r >= rows) return;
    const uint16_t* wr = W + static_cast<size_t>(r) * cols;
    float acc = 0.f;
    for (uint32_t c = lane; c < cols; c += WAVE) acc = fmaf(bf16_to_f32(wr[c]), x[c], acc);
    acc = wave_sum(acc);
    if (lane == 0) out[r] = acc;
}

hipError_t launch_matvec_bf16(const uint16_t* W, const float* x, float* out, uint32_t rows, uint32_t cols,
                              hipStream_t s)
{
    if (rows == 0 || cols == 0) return hipErrorInvalidValue;
    launch_kernel(k_matvec_bf16, dim3((rows + 3) / 4), dim3(256), s, W, x, out, rows, cols);
    return hipGetLastError();
}

}  // namespace smoe
