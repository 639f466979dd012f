// fake_hip.cpp -- a HIP runtime and kernel launchers without a device, for tests
// of the host side of the C ABI (csrc/bridge.cpp) on the CPU: device memory is
// bookkeeping only (an address range per allocation, an optional budget), host
// memory is real, launches are recorded and do nothing.  Compiled together with
// bridge.cpp by tests/test_bridge_host.py; the fake_* functions steer it.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

#include "kernels.hpp"

namespace {

struct State {
    std::map<uintptr_t, size_t> dev, host;   // live allocations
    uintptr_t next = uintptr_t(1) << 44;
    size_t budget = ~size_t(0), live = 0;
    bool capturing = false;
    uint64_t mallocs = 0, frees = 0, host_mallocs = 0, host_frees = 0, syncs = 0, failed = 0;
    std::string fail;                        // launcher that fails next
    // the last prefill pass
    uintptr_t x_hi = 0, y = 0;
    uint32_t T = 0;
    uint64_t routes = 0, permutes = 0, permutes_seg = 0;
};
State& st()
{
    static State s;
    return s;
}

// what launch_kernel does with the timer: every dispatch takes its events
hipError_t dispatch(const char* name, int n = 1)
{
    if (st().fail == name) {
        st().fail.clear();
        return hipErrorLaunchFailure;
    }
    for (int i = 0; i < n; ++i) (void)smoe::dispatch_timer().take();
    return hipSuccess;
}

}  // namespace

// ---- steering ---------------------------------------------------------------
extern "C" {
void fake_budget(size_t bytes) { st().budget = bytes; }
void fake_capturing(int on) { st().capturing = on != 0; }
void fake_fail(const char* launcher) { st().fail = launcher; }
uint64_t fake_count(const char* what)
{
    const std::string w = what;
    State& s = st();
    if (w == "mallocs") return s.mallocs;
    if (w == "frees") return s.frees;
    if (w == "host_mallocs") return s.host_mallocs;
    if (w == "host_frees") return s.host_frees;
    if (w == "syncs") return s.syncs;
    if (w == "failed") return s.failed;
    if (w == "live") return s.live;
    if (w == "host_allocations") return s.host.size();
    if (w == "allocations") return s.dev.size();
    if (w == "x_hi") return s.x_hi;
    if (w == "y") return s.y;
    if (w == "T") return s.T;
    if (w == "routes") return s.routes;
    if (w == "permutes") return s.permutes;
    if (w == "permutes_seg") return s.permutes_seg;
    return ~0ull;
}
uint32_t fake_unit_cap(uint32_t P, uint32_t u64, uint32_t u32, uint32_t tiles)
{
    return smoe::unit_cap(P, u64, u32, tiles);
}
uint32_t fake_unit_slots(uint32_t P, uint32_t E, uint32_t tiles) { return smoe::unit_slots(smoe::max_units(P, E, tiles)); }
void fake_unit_share(uint32_t x, uint32_t n_long, uint32_t n_short, uint32_t* out)
{
    const smoe::UnitShare u = smoe::unit_share(x, n_long, n_short);
    out[0] = u.l0, out[1] = u.nl, out[2] = u.s0, out[3] = u.ns;
}
uint64_t fake_unit_records(uint32_t P, uint32_t E) { return smoe::unit_records(P, E); }
int fake_lds_weights(uint32_t P, uint32_t E, uint32_t tiles) { return smoe::lds_weights(P, E, tiles); }
int fake_attn_wide(uint32_t heads, uint32_t kv_heads, uint32_t head_dim, uint32_t valid)
{
    return smoe::attn_wide({head_dim, heads, kv_heads, kv_heads * head_dim, valid, 1.0f}, valid);
}
int fake_is_live(uint64_t p) { return st().dev.count(static_cast<uintptr_t>(p)) != 0; }

// ---- the runtime --------------------------------------------------------------
hipError_t hipMalloc(void** p, size_t n)
{
    State& s = st();
    if (s.capturing) return hipErrorStreamCaptureUnsupported;
    if (n > s.budget - std::min(s.budget, s.live)) {
        ++s.failed;
        return hipErrorOutOfMemory;
    }
    ++s.mallocs;
    *p = reinterpret_cast<void*>(s.next);
    s.dev[s.next] = n;
    s.next += (n + 4095) / 4096 * 4096;
    s.live += n;
    return hipSuccess;
}
hipError_t hipFree(void* p)
{
    State& s = st();
    const auto it = s.dev.find(reinterpret_cast<uintptr_t>(p));
    if (it == s.dev.end()) std::abort();      // not ours, or freed twice
    ++s.frees;
    s.live -= it->second;
    s.dev.erase(it);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned int)
{
    *p = std::malloc(n);
    st().host[reinterpret_cast<uintptr_t>(*p)] = n;
    ++st().host_mallocs;
    return hipSuccess;
}
hipError_t hipHostFree(void* p)
{
    if (!st().host.erase(reinterpret_cast<uintptr_t>(p))) std::abort();
    ++st().host_frees;
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemset(void*, int, size_t) { return hipSuccess; }
hipError_t hipMemcpy(void* dst, const void*, size_t n, hipMemcpyKind kind)
{
    if (kind == hipMemcpyDeviceToHost) std::memset(dst, 0, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind kind, hipStream_t)
{
    return hipMemcpy(dst, src, n, kind);
}
hipError_t hipStreamSynchronize(hipStream_t)
{
    ++st().syncs;
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipStreamSynchronize(nullptr); }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned int)
{
    *s = reinterpret_cast<hipStream_t>(uintptr_t(64));
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* c)
{
    *c = st().capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned int)
{
    static uintptr_t n = 64;
    *e = reinterpret_cast<hipEvent_t>(n += 64);
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return dispatch("event_record", 0); }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t)
{
    *ms = 1.0f;                               // every dispatch takes 1 ms
    return hipSuccess;
}
hipError_t hipGetDeviceCount(int* n)
{
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetDevice(int* d)
{
    *d = 0;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "fake"; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t*, const void*) { return hipErrorInvalidValue; }
}

// ---- the launchers --------------------------------------------------------------
namespace smoe {

DispatchTimer& dispatch_timer()
{
    static DispatchTimer t;
    return t;
}
uint64_t* static_scratch_setup() { return nullptr; }
bool deal_probe() { return true; }
bool layer_supported(const MoeDims&, const LayerDesc&) { return false; }
bool chain_supported(const MoeDims&, const LayerDesc*, uint32_t) { return false; }
size_t attn_scratch_bytes(const AttnDims& a) { return size_t(a.num_heads) * 64 * (2 + a.head_dim) * 4; }

hipError_t launch_moe_up(const MoeDims&, const LayerDesc&, const float*, uint32_t, uint64_t*, float*, uint32_t*, float*,
                         ExpertPtrs*, uint32_t*, hipStream_t)
{
    return dispatch("moe_up");
}
hipError_t launch_down_combine(const MoeDims&, const ExpertPtrs*, const float*, const float*, float*, uint64_t*,
                               uint32_t, hipStream_t)
{
    return dispatch("moe_down");
}
hipError_t launch_moe_layer(const MoeDims&, const LayerDesc&, float*, uint64_t*, uint32_t*, float*, uint32_t*, hipStream_t)
{
    return dispatch("moe_layer");
}
hipError_t launch_moe_chain(const MoeDims&, const LayerDesc*, uint32_t, float*, uint64_t*, float*, uint32_t*, uint32_t*,
                            float*, uint32_t*, hipStream_t)
{
    return dispatch("chain");
}
hipError_t launch_stage_in(const float*, float*, uint32_t, hipStream_t) { return dispatch("stage_in", 0); }
hipError_t launch_gate_up(const MoeDims&, const ExpertTable&, uint32_t, const float*, float*, uint32_t, hipStream_t)
{
    return dispatch("gate_up");
}
hipError_t launch_down_slots(const MoeDims&, const ExpertTable&, uint32_t, const float*, uint32_t, float*, uint32_t,
                             hipStream_t)
{
    return dispatch("down");
}
hipError_t launch_gate_up_tokens(const MoeDims&, const ExpertPtrs&, const float*, float*, uint32_t, hipStream_t)
{
    return dispatch("gate_up_tokens");
}
hipError_t launch_down_tokens(const MoeDims&, const ExpertPtrs&, const float*, float*, uint32_t, hipStream_t)
{
    return dispatch("down_tokens");
}
hipError_t launch_topk(const float*, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t*, float*, hipStream_t)
{
    return dispatch("topk");
}
hipError_t launch_matvec_bf16(const uint16_t*, const float*, float*, uint32_t, uint32_t, hipStream_t)
{
    return dispatch("matvec", 0);
}
hipError_t launch_gemv_bf16(const GemvGroup&, hipStream_t) { return dispatch("gemv"); }
hipError_t launch_attention(const AttnDims&, const float*, const float*, const float*, const uint16_t*, const uint16_t*,
                            const float*, const float*, float*, float*, uint32_t, uint32_t, void*, float*, hipStream_t)
{
    return dispatch("attention", 2);          // attention and combine
}
hipError_t launch_route(const MoeDims&, const LayerDesc&, const float*, uint32_t T, uint16_t* x_hi, uint16_t*, float*,
                        uint32_t*, float*, float*, uint32_t*, hipStream_t)
{
    st().x_hi = reinterpret_cast<uintptr_t>(x_hi);
    st().T = T;
    ++st().routes;
    return dispatch("route");
}
hipError_t launch_split_rows(const float*, uint32_t, uint32_t, uint16_t*, uint16_t*, float*, hipStream_t)
{
    return dispatch("split");
}
hipError_t launch_permute(const uint32_t*, const float*, uint32_t, uint32_t, uint32_t, uint32_t*, uint32_t*, uint32_t*,
                          float*, uint32_t*, uint32_t*, const UnitLists&, uint32_t*, hipStream_t)
{
    ++st().permutes;
    return dispatch("permute");
}
hipError_t launch_permute_seg(const uint32_t*, uint32_t P, uint32_t E, uint32_t*, const UnitLists&, uint32_t*, uint32_t*,
                              hipStream_t)
{
    ++st().permutes_seg;
    return dispatch("permute_seg", perm_segments(P, E) > 1 ? 2 : 1);
}
hipError_t launch_grouped_gate_up(const MoeDims&, const LayerDesc&, uint32_t, const UnitLists&, const uint32_t*,
                                  const uint16_t*, const uint16_t*, const float*, float*, hipStream_t)
{
    return dispatch("grouped_gate_up");
}
hipError_t launch_grouped_down(const MoeDims&, const LayerDesc&, uint32_t, const UnitLists&, const uint32_t*,
                               const uint16_t*, const uint16_t*, const float*, float* y, hipStream_t)
{
    st().y = reinterpret_cast<uintptr_t>(y);
    return dispatch("grouped_down");
}
hipError_t launch_combine_pairs(const float*, const float*, uint32_t, uint32_t, uint32_t, float*, hipStream_t)
{
    return dispatch("combine");
}
hipError_t launch_stream_read(const void*, uint64_t, uint32_t*, hipStream_t) { return dispatch("stream_read"); }
hipError_t launch_synth_normal(float*, uint64_t, uint64_t, uint64_t, float, hipStream_t) { return hipSuccess; }
hipError_t launch_synth_bf16(uint16_t*, uint64_t, uint64_t, uint64_t, float, hipStream_t) { return hipSuccess; }
hipError_t launch_quantize_q4(const float*, uint64_t, uint32_t, uint8_t*, uint16_t*, hipStream_t) { return hipSuccess; }
hipError_t launch_quantize_q4_min(const float*, uint64_t, uint32_t, uint8_t*, uint16_t*, uint16_t*, hipStream_t)
{
    return hipSuccess;
}
hipError_t launch_synth_pool(uint8_t*, uint32_t, uint32_t, uint32_t, uint64_t, uint32_t, uint32_t, uint32_t,
                             const uint64_t*, uint64_t, float, uint32_t, hipStream_t)
{
    return hipSuccess;
}

}  // namespace smoe
