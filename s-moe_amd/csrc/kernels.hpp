// kernels.hpp -- host-side launchers of the gfx950 MoE kernels (internal to
// libsmoe_hip.so; the public surface is include/smoe_hip.h).
#pragma once

#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace smoe {

// largest expert count a top-k wave handles (8 positions per lane)
constexpr int SMOE_TOPK_MAX_N = 512;
constexpr int SMOE_TOPK_MAX_K = 16;

// Events that time the next kernel dispatches of this thread, a pair for each
// (a launcher may dispatch twice): while pairs are left, the launchers dispatch
// through hipExtLaunchKernel, which records `start` when the kernel begins
// executing and `stop` when it completes (the dispatch's own timestamps, no
// marker packets around it).  Set only around eager launches by the profiling
// path of the C ABI.
struct DispatchTimer {
    static constexpr int MAX = 2;             // dispatches of one launcher
    struct Pair {
        hipEvent_t start = nullptr;
        hipEvent_t stop = nullptr;
    };
    Pair pair[MAX];
    int n = 0;                                // pairs given
    int used = 0;                             // pairs that dispatches have taken
    Pair take() { return used < n ? pair[used++] : Pair{}; }
};
DispatchTimer& dispatch_timer();

template <typename... KArgs, typename... Args>
inline void launch_kernel_lds(void (*k)(KArgs...), dim3 grid, dim3 block, uint32_t lds, hipStream_t s, Args... args)
{
    const DispatchTimer::Pair t = dispatch_timer().take();
    if (t.start)
        hipExtLaunchKernelGGL(k, grid, block, lds, s, t.start, t.stop, 0, static_cast<KArgs>(args)...);
    else
        hipLaunchKernelGGL(k, grid, block, lds, s, static_cast<KArgs>(args)...);
}

template <typename... KArgs, typename... Args>
inline void launch_kernel(void (*k)(KArgs...), dim3 grid, dim3 block, hipStream_t s, Args... args)
{
    launch_kernel_lds(k, grid, block, 0u, s, args...);
}

// Routing exchange of one token: LL_COPIES copies of its E logit words (flag
// in the high half), ll_copy_words(E) words apart (> 4 KB), so the waves that
// poll them spread over several memory channels instead of queueing on one.
constexpr uint32_t LL_COPIES = 8;
__host__ __device__ constexpr uint32_t ll_copy_words(uint32_t E) { return (E > 512u ? E : 512u) + 32u; }
__host__ __device__ constexpr size_t ll_token_words(uint32_t E) { return size_t(LL_COPIES) * ll_copy_words(E); }

// Six tensor pointers of one expert plus the scratch slot its results use.
struct ExpertPtrs {
    const uint8_t*  pg;
    const uint16_t* sg;
    const uint8_t*  pu;
    const uint16_t* su;
    const uint8_t*  pd;
    const uint16_t* sd;
    uint32_t        slot;
    uint32_t        pad_;
};

// The experts of one reference-surface dispatch (SMOE_MAX_ACTIVE), a kernel argument.
struct ExpertTable {
    static constexpr uint32_t MAX = 16;
    ExpertPtrs e[MAX];
};

struct MoeDims {
    uint32_t D, E, K, I, group, norm_topk;
    uint32_t quant = 0;   // SMOE_QUANT_*: 0 fp16 absmax (SMOE-Q4), 1 bf16 scale + bf16 min
};

struct LayerDesc {
    const uint16_t* norm_w;
    const uint16_t* router_w;
    const uint8_t*  experts;
    uint64_t        stride;
    uint64_t        off[6];   // gate p, gate s, up p, up s, down p, down s
};

// ---- decode, one token (moe_decode.hip) ----------------------------------
// Router + softmax/top-k (+renorm) + gate/up/SiLU of the selected experts:
// h [T x K x I]; publishes ids/w [T x K] and the expert table [T x K].
// ll [T x (E+1)] must be zero on entry (launch_down_combine re-arms it);
// err receives 1 if the routing exchange timed out.
hipError_t launch_moe_up(const MoeDims& d, const LayerDesc& L, const float* hidden, uint32_t n_tok, uint64_t* ll,
                         float* h, uint32_t* ids, float* w, ExpertPtrs* tbl, uint32_t* err, hipStream_t s);
// n floats (a multiple of 4) from pinned host memory to the device
hipError_t launch_stage_in(const float* src, float* dst, uint32_t n, hipStream_t s);
// reference surface, one vector: h[slot * h_stride + row] = silu(gate.x) * (up.x)
// for n_exp table entries, and out[slot * out_stride + row] = down_slot . h_slot
hipError_t launch_gate_up(const MoeDims& d, const ExpertTable& tbl, uint32_t n_exp, const float* x, float* h,
                          uint32_t h_stride, hipStream_t s);
hipError_t launch_down_slots(const MoeDims& d, const ExpertTable& tbl, uint32_t n_exp, const float* h,
                             uint32_t h_stride, float* out, uint32_t out_stride, hipStream_t s);
// reference surface, one expert and n_tok vectors: h [n_tok x I] from x [n_tok x D],
// out [n_tok x D] from h (rows multiples of 32, groups of 32, 64 or 128)
hipError_t launch_gate_up_tokens(const MoeDims& d, const ExpertPtrs& e, const float* x, float* h, uint32_t n_tok,
                                 hipStream_t s);
hipError_t launch_down_tokens(const MoeDims& d, const ExpertPtrs& e, const float* h, float* out, uint32_t n_tok,
                              hipStream_t s);
// hidden[t][row] += sum_r w[t][r] * (down_r . h[t][r])  (weighted combine + residual);
// zeroes ll [T x (E+1)] for the next launch_moe_up
hipError_t launch_down_combine(const MoeDims& d, const ExpertPtrs* tbl, const float* h, const float* w,
                               float* hidden, uint64_t* ll, uint32_t n_tok, hipStream_t s);
// ---- decode, one token, one launch (moe_layer.hip) -----------------------
// Exchange-word tags of the one-launch decode kernels.  The epoch word holds
// a count e in [0, TAG_PERIOD); the words of layer l of a launch that read e
// carry tag_at(e, l) = ((e + l) mod TAG_PERIOD) + 1, and the launch leaves
// epoch_after(e, n_layers) behind.  Tags therefore run through 1 .. 2^32 - 1
// and wrap from 2^32 - 1 to 1: never 0 (every word's value at allocation),
// and two consecutive layers, in one launch or across launches, never share
// one.  Any 32-bit value read from the word is reduced first, so a word
// holding 2^32 - 1 counts as 0.
constexpr uint32_t TAG_PERIOD = 0xFFFFFFFFu;
__host__ __device__ constexpr uint32_t tag_mod(uint64_t s)
{
    // s mod (2^32 - 1): 2^32 is 1 modulo the period, so fold the high word in
    const uint64_t f = (s & 0xFFFFFFFFull) + (s >> 32);   // < 2^33
    const uint64_t g = (f & 0xFFFFFFFFull) + (f >> 32);   // <= 2^32
    return static_cast<uint32_t>(g >= TAG_PERIOD ? g - TAG_PERIOD : g);
}
__host__ __device__ constexpr uint32_t tag_at(uint32_t epoch, uint32_t l)
{
    return tag_mod(static_cast<uint64_t>(epoch) + l) + 1u;
}
__host__ __device__ constexpr uint32_t epoch_after(uint32_t epoch, uint32_t n_layers)
{
    return tag_mod(static_cast<uint64_t>(epoch) + n_layers);
}
// Exchange words of the one-launch layer: word 0 holds the epoch (above),
// then 8 logit copies of lx_pad(E) words, 8 h copies of lx_pad(I) words and
// 8 rank partials of lx_pad(D) words.  Zero once at allocation; never
// re-armed (a launch that times out leaves them to be cleared by the host).
constexpr uint32_t LX_HEAD = 64;
constexpr uint32_t LX_MAX_I = 2048;
__host__ __device__ constexpr uint32_t lx_pad(uint32_t n) { return ((n + 63u) & ~63u) + 64u; }
__host__ __device__ constexpr size_t lx_words(uint32_t D, uint32_t E, uint32_t I)
{
    return LX_HEAD + 8ull * (lx_pad(E) + lx_pad(I) + lx_pad(D));
}
// Checks once per device (synchronously, outside stream capture) that blocks
// are dealt round-robin over the 8 XCDs, which the one-launch layer kernels
// rely on; later calls return the cached answer.
bool deal_probe();
// true when k == 8, the shape's grid fits on the device at once, the layer's
// tensors are 16-byte aligned and the device deals blocks round-robin (as
// deal_probe found; false before it ran)
bool layer_supported(const MoeDims& d, const LayerDesc& L);
// the whole MoE block of one token: hidden [D] += MoE(RMSNorm(hidden));
// ids/w [K] receive the routing; err bit 0 reports an exchange time-out
hipError_t launch_moe_layer(const MoeDims& d, const LayerDesc& L, float* hidden, uint64_t* lx, uint32_t* ids,
                            float* w, uint32_t* err, hipStream_t s);
// Every layer of a decode step in one launch with k_moe_layer's schedule per
// layer.  xch: chain_xch_words(D, E, I) exchange words; hcopy [8 x D] floats;
// cnt chain_cnt_words() words (per-XCD row-block flags, then an abort word);
// all zero at allocation and never re-armed
// (calls on one set must not overlap).  layers_dev: the layer table in device
// memory; ids/w [n_layers x K].
constexpr uint32_t CHAIN_FLAGS = 256;       // row-block flags per XCD (n_down <= 256)
__host__ __device__ constexpr size_t chain_xch_words(uint32_t D, uint32_t E, uint32_t I)
{
    return lx_words(D, E, I) + 8ull * lx_pad(D);
}
constexpr size_t chain_cnt_words() { return 8 * CHAIN_FLAGS + 64; }
bool chain_supported(const MoeDims& d, const LayerDesc* layers_host, uint32_t n_layers);
hipError_t launch_moe_chain(const MoeDims& d, const LayerDesc* layers_dev, uint32_t n_layers, float* hidden,
                            uint64_t* xch, float* hcopy, uint32_t* cnt, uint32_t* ids, float* w, uint32_t* err,
                            hipStream_t s);
// softmax + top-k over rows of scores (scout.cpp:77-123)
hipError_t launch_topk(const float* scores, uint32_t rows, uint32_t n, uint32_t k,
                       uint32_t norm, uint32_t* ids, float* w, hipStream_t s);


// out [rows] = W [rows x cols] bf16 . x [cols] (reference-surface dense GEMV)
hipError_t launch_matvec_bf16(const uint16_t* W, const float* x, float* out, uint32_t rows, uint32_t cols,
                              hipStream_t s);

// ---- dense trunk (trunk.hip) ---------------------------------------------
// up to GEMV_MAX independent y = W x (bf16 W [rows x cols], fp32 x, y) in one
// launch; cols % 8 == 0, cols <= GEMV_MAX_COLS, W and x 16-byte aligned
constexpr uint32_t GEMV_MAX = 8;
constexpr uint32_t GEMV_MAX_COLS = 16384;
struct GemvGroup {
    const uint16_t* w[GEMV_MAX];
    const float* x[GEMV_MAX];
    float* y[GEMV_MAX];
    uint32_t rows[GEMV_MAX], cols[GEMV_MAX], block0[GEMV_MAX];
    uint32_t count;
};
hipError_t launch_gemv_bf16(const GemvGroup& g, hipStream_t s);

// single-token decode attention over a KV ring of ctx positions: one fused
// launch (QK norm + RoPE + KV append, attention per (KV head, query-head
// group, context split) with an online softmax), and with several splits a
// combine launch, into attn_out [q_dim].  head_dim 64, 128 or 256.
constexpr uint32_t ATTN_MAX_SPLITS = 64;
struct AttnDims {
    uint32_t head_dim, num_heads, num_kv_heads, kv_dim, ctx;
    float scale;
};
struct AttnPlan {
    bool wide;          // k_attn_wide
    uint32_t gb;        // query heads per block (16, or a power of two <= 8)
    uint32_t n_sub;     // blocks per KV head along the query heads
    uint32_t splits;    // context splits
    uint32_t chunk;     // positions per split
};
constexpr int AT_MAX_GB = 8;      // k_attn_decode: query heads per block,
constexpr int AT_MAX_GHD = 1024;  // times head_dim
constexpr int AW_HEADS = 16;      // k_attn_wide: query heads per block (MFMA columns)
// query heads per block of k_attn_decode
constexpr uint32_t attn_group(const AttnDims& a)
{
    const uint32_t G = a.num_heads / a.num_kv_heads;
    uint32_t gb = 1;
    while (gb < G && gb < static_cast<uint32_t>(AT_MAX_GB) && gb * 2 * a.head_dim <= AT_MAX_GHD) gb *= 2;
    return gb;
}
// The MFMA kernel (k_attn_wide) reads each K and V row once for all query heads of
// a KV head, k_attn_decode once per block of up to eight.  Long contexts with more
// than eight: 16 heads of 128 over 32768 positions 80 -> 59 us for the layer, 64
// heads of 256 over 4 KV heads 195 -> 91.  Over 1000 positions, where the launches'
// latencies decide, it loses (39.5 against 38.7; ten of 256 over 2048 27.1 against
// 24.0), at 3000 the two are even, and with eight heads or fewer its columns are
// half or more empty (8 heads over 32768 positions 39.3 against 41.8, one head 31.5
// against 30.0).  With up to 64 splits it has 64 blocks for each 16 query heads of a
// KV head, and half the waves a block at head_dim 256.  One such column of 256:
// slower at every length (10 heads 20.0 against 23.0 us at 4096 positions, 43.8
// against 59.8 at 32768).  One or two columns, where k_attn_decode's blocks have no
// idle heads: from 8192 positions on (16 heads of 128 over one KV head 19.4 / 20.3
// at 4096, 20.1 / 20.3 at 6000, 21.6 / 20.8 at 8192; 32 of 256 over two 33.5 / 34.6,
// 37.9 / 38.5, 42.4 / 39.8; with idle heads, 20 of 256 over two, 29.4 / 27.6 at
// 4096); heads of 64 from 4096 on (17.3 / 16.5).
constexpr bool attn_wide(const AttnDims& a, uint32_t valid)
{
    const uint32_t G = a.num_heads / a.num_kv_heads, columns = a.num_kv_heads * ((G + AW_HEADS - 1) / AW_HEADS);
    if (G <= static_cast<uint32_t>(AT_MAX_GB) || (a.head_dim > 128 && columns == 1)) return false;
    return valid >= (a.head_dim > 64 && columns <= 2 && G % attn_group(a) == 0 ? 8192u : 4096u);
}
AttnPlan attn_plan(const AttnDims& a, uint32_t valid);
// scratch of the launch: per-(head, split) partials
size_t attn_scratch_bytes(const AttnDims& a);
hipError_t launch_attention(const AttnDims& a, const float* q, const float* k, const float* v,
                            const uint16_t* q_norm_w, const uint16_t* k_norm_w, const float* rope_cos,
                            const float* rope_sin, float* k_cache, float* v_cache, uint32_t slot, uint32_t valid,
                            void* scratch, float* attn_out, hipStream_t s);

// ---- prefill, T token rows (moe_prefill.hip) -----------------------------
// RMSNorm + router + top-k for T tokens: the normed rows as f16 planes
// x_hi/x_lo [T x D] with row scales x_sc [T] (as launch_split_rows writes
// them), ids/w [T x K].  logits [T x E] and counters [T] (zero at allocation;
// every launch adds a multiple of 4) serve the short-batch form; with either
// null every token group runs in one block.
hipError_t launch_route(const MoeDims& d, const LayerDesc& L, const float* hidden, uint32_t T, uint16_t* x_hi,
                        uint16_t* x_lo, float* x_sc, uint32_t* ids, float* w, float* logits, uint32_t* counters,
                        hipStream_t s);
// Per row of src [rows x cols]: f16 hi/lo planes of x * 2^-e (|x| < 2^e over
// the row) and scale[row] = 2^e.
hipError_t launch_split_rows(const float* src, uint32_t rows, uint32_t cols, uint16_t* hi, uint16_t* lo,
                             float* scale, hipStream_t s);
// The grouped GEMMs' work lists, one for gate/up and one for down: units of up to
// cap (64 or 32) pairs of one expert, u64 or u32 of them, a block for each unit and
// each of the launch's row tiles.  Units of 32 run a long expert's passes side by
// side but stream and convert its weights once more each, so they are worth it
// where they cost no more than the CUs that would otherwise be idle: where the
// longest XCD's share still gives its 32 CUs at most one block each; and where
// units of 64 are over that too, up to two blocks a CU if there are few more of
// 32 (a few long experts) or those of 64 are mostly full.  Kernel times in us with
// units of 64 / of 32:
//   one block a CU at most   16 experts, 23 units of 32, 10 tiles  44.5 / 41.2
//                            8 experts, 23, 6                      36.7 / 26.8
//                            64, 31, 5 (skewed)                    22.9 / 17.4
//   more                     16, 32, 10                            55.7 / 63.5
//                            32, 33, 8                             15.8 / 22.0
//                            64, 132, 7                            62.4 / 83.4
//   62 for 57 units, 6 tiles (64 Zipf-routed tokens of 128 experts)  43.3 / 39.2
//   77 for 45 units of 44 pairs, 6 tiles                           59.1 / 46.0
__host__ __device__ constexpr uint32_t unit_cap(uint32_t P, uint32_t u64, uint32_t u32, uint32_t tiles)
{
    const uint32_t b64 = (u64 + 7u) / 8u * tiles, b32 = (u32 + 7u) / 8u * tiles;   // blocks of an XCD
    if (b32 <= 32u) return 32u;
    return b64 > 32u && b32 <= 64u && (8u * u32 <= 9u * u64 || P >= 40u * u64) ? 32u : 64u;
}
constexpr uint32_t max_units(uint32_t P, uint32_t E, uint32_t tiles)
{
    const uint32_t experts = E < P ? E : P, u64 = P / 64 + experts, u32 = P / 32 + experts;
    const uint32_t two = 64 / tiles * 8, m32 = u32 < two ? u32 : two;   // (units of 32: two blocks a CU at most)
    return u64 > m32 ? u64 : m32;
}
// XCD x's share of a work list: consecutive long units, then consecutive short ones.
// The XCDs with one short unit more follow those with one long unit more, so that no
// share is over an eighth of the units rounded up.  A share one unit over that cost
// 62 units of 12 tiles 86 us for 76.
struct UnitShare {
    uint32_t l0, nl;   // first long unit, number
    uint32_t s0, ns;   // first short unit, number
};
__host__ __device__ constexpr UnitShare unit_share(uint32_t x, uint32_t n_long, uint32_t n_short)
{
    const uint32_t a = n_long & 7u, b = n_short & 7u, y = (x - a) & 7u;
    return {x * (n_long >> 3) + (x < a ? x : a), (n_long >> 3) + (x < a ? 1u : 0u),
            y * (n_short >> 3) + (y < b ? y : b), (n_short >> 3) + (y < b ? 1u : 0u)};
}
// records of a work list: the eight shares, each as long as the longest can be
constexpr uint32_t unit_slots(uint32_t units) { return (units + 7u) / 8u * 8u; }
struct UnitLists {
    uint4* units = nullptr;       // [slots[0] + slots[1]], null: none
    uint32_t tiles[2] = {1, 1};   // row tiles of gate/up and of down
    uint32_t slots[2] = {0, 0};
};
inline UnitLists unit_lists(const MoeDims& d, uint32_t P, uint4* units)
{
    UnitLists l;
    l.units = units;
    l.tiles[0] = (d.I + 127u) / 128u;
    l.tiles[1] = (d.D + 255u) / 256u;
    for (int i = 0; i < 2; ++i) l.slots[i] = unit_slots(max_units(P, d.E, l.tiles[i]));
    return l;
}
// Whether a launch of the grouped GEMMs takes k_grouped_mm though k_grouped_reg could
// run it: where its blocks are at most one a CU, half of the waves that a CU holds
// of k_grouped_reg would be missing.  The host knows of the units that there is at
// most one for every expert with a pair and one more for every 64 pairs.  Kernel
// times in us, k_grouped_reg / k_grouped_mm: 16 experts, 10 tiles of 3072 columns, 64
// tokens 32.1 / 29.0; 8 experts, 4 and 16 tiles, 60 tokens (down) 21.9 / 20.8; one
// expert, 6 tiles, 16 tokens 21.4 / 18.7; over one a CU 60 experts, 6 tiles 26.0 /
// 28.0, and 68 units of 64 pairs, 4 tiles 34.3 / 42.6.
constexpr bool lds_weights(uint32_t P, uint32_t E, uint32_t tiles)
{
    return ((E < P ? E : P) + P / 64) * tiles <= 256;
}
// what unit_lists takes at most
constexpr size_t unit_records(uint32_t P, uint32_t E) { return 2 * size_t(unit_slots(P / 32 + (E < P ? E : P))); }
// Stable counting sort of the P pairs by expert: offsets [E+1],
// sorted_pairs [P] (pair = token * K + rank); sorted_tokens, sorted_w,
// union_ids [E], union_size [1] optional (nullptr), and the work lists.  Bad ids
// set err bit 1.
constexpr size_t PERMUTE_MAX_LDS = 48 * 1024;
constexpr size_t permute_lds_bytes(uint32_t P, uint32_t E)
{
    return (size_t((P + 63) / 64) * E + 3 * size_t(E) + 1) * sizeof(uint32_t);
}
hipError_t launch_permute(const uint32_t* ids, const float* w, uint32_t P, uint32_t K, uint32_t E, uint32_t* offsets,
                          uint32_t* sorted_pairs, uint32_t* sorted_tokens, float* sorted_w, uint32_t* union_ids,
                          uint32_t* union_size, const UnitLists& lists, uint32_t* err, hipStream_t s);
// The same sorted pairs and work lists in segments, one workgroup each, for any P
// (seg_cnt [perm_segments(P, E) x E]).
__host__ __device__ constexpr uint32_t perm_seg_chunks(uint32_t E) { return E <= 256 ? 32u : 16u; }
constexpr uint32_t perm_segments(uint32_t P, uint32_t E)
{
    return (P + 64u * perm_seg_chunks(E) - 1) / (64u * perm_seg_chunks(E));
}
hipError_t launch_permute_seg(const uint32_t* ids, uint32_t P, uint32_t E, uint32_t* sorted_pairs,
                              const UnitLists& lists, uint32_t* seg_cnt, uint32_t* err, hipStream_t s);
// Whether a batch of several segments is permuted in one workgroup all the same:
// one launch instead of two, but one CU's time for all the pairs.  Call times in
// us of one workgroup / both segment kernels at 128 experts x top-8: 260 tokens
// 134.7 / 135.8, 400 151.1 / 151.8, 512 160.2 / 160.2, 640 188.3 / 187.4, 736 215.1
// / 213.2; 32 x top-4: 700 tokens 116.7 / 117.5, 1500 192.1 / 191.3; 8 x top-2:
// 1500 52.0 / 53.1, 4000 86.8 / 85.6; 512 x top-8, 150 tokens 118.0 / 119.5.  (The
// kernels' own times say more, 7.7 against 9.5 us at 512 tokens: the second of two
// short launches hides part of the first one's.)  One segment is permuted by
// k_perm_scatter alone.
constexpr bool permute_in_one(uint32_t P, uint32_t E)
{
    return perm_segments(P, E) > 1 && P <= 4096 && permute_lds_bytes(P, E) <= PERMUTE_MAX_LDS;
}
// Grouped expert GEMMs over the permuted pairs (MFMA f16, hi/lo activations):
// h [P x I] = silu(x G^T) * (x U^T); y [P x D] = h Dn^T, over the permute's
// work lists.
hipError_t launch_grouped_gate_up(const MoeDims& d, const LayerDesc& L, uint32_t P, const UnitLists& lists,
                                  const uint32_t* sorted_pairs, const uint16_t* x_hi,
                                  const uint16_t* x_lo, const float* x_scale, float* h, hipStream_t s);
hipError_t launch_grouped_down(const MoeDims& d, const LayerDesc& L, uint32_t P, const UnitLists& lists,
                               const uint32_t* sorted_pairs, const uint16_t* h_hi,
                               const uint16_t* h_lo, const float* h_scale, float* y, hipStream_t s);
// hidden[t] += sum_r w[t][r] * y[t*K + r] (rank order).
hipError_t launch_combine_pairs(const float* y, const float* w, uint32_t T, uint32_t K, uint32_t D, float* hidden,
                                hipStream_t s);

// ---- static scratch of smoe_hip_moe_decode_static (decode_static.hip) -----
// Takes the current device's address of the file-scope scratch array and
// clears it, once per device (synchronous; outside stream capture).
uint64_t* static_scratch_setup();

// ---- measurement (probe.hip) ----------------------------------------------
// Streams `bytes` (a multiple of 16) from src with non-temporal 128-bit loads;
// folds what it read into *sink.
hipError_t launch_stream_read(const void* src, uint64_t bytes, uint32_t* sink, hipStream_t s);

// ---- synthetic generator / quantizer (synth.hip) -------------------------
hipError_t launch_synth_normal(float* out, uint64_t n, uint64_t seed, uint64_t stream,
                               float stddev, hipStream_t s);
hipError_t launch_synth_bf16(uint16_t* out, uint64_t n, uint64_t seed, uint64_t stream,
                             float stddev, hipStream_t s);
hipError_t launch_quantize_q4(const float* w, uint64_t n, uint32_t group, uint8_t* packed,
                              uint16_t* scales, hipStream_t s);
// the scale+min format: scales and mins [n / group] bf16 bits
hipError_t launch_quantize_q4_min(const float* w, uint64_t n, uint32_t group, uint8_t* packed,
                                  uint16_t* scales, uint16_t* mins, hipStream_t s);
// quant: SMOE_QUANT_*; with the scale+min format each matrix's mins follow
// its D*I/group scales
hipError_t launch_synth_pool(uint8_t* base, uint32_t first_layer, uint32_t n_layers,
                             uint32_t n_experts, uint64_t stride, uint32_t D, uint32_t I,
                             uint32_t group, const uint64_t* off6, uint64_t seed,
                             float stddev, uint32_t quant, hipStream_t s);

}  // namespace smoe
