"""The host side of the C ABI (csrc/bridge.cpp) on the CPU: compiled against a
HIP runtime and launchers that only keep books (fake_hip.cpp), so that memory
that runs out, launches that fail and stream capture can be forced."""
import ctypes as C
import os
import re
import shutil
import subprocess

import numpy as np
import pytest

import smoe_amd

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SHAPE_30B = dict(d_model=2048, n_experts=128, top_k=8, d_ff=768)
DEV = 1 << 20        # stands for any device address


@pytest.fixture(scope="module")
def built(tmp_path_factory):
    cxx = "/opt/rocm/llvm/bin/clang++"
    cxx = cxx if os.path.exists(cxx) else shutil.which("clang++")
    so = str(tmp_path_factory.mktemp("fake") / "libbridge_fake.so")
    r = subprocess.run(
        [cxx, "-std=c++17", "-O1", "-shared", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
         "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(ROOT, "s-moe_amd", "csrc"),
         os.path.join(ROOT, "s-moe_amd", "csrc", "bridge.cpp"), os.path.join(ROOT, "tests", "fake_hip.cpp"),
         "-Wl,-Bsymbolic", "-o", so], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return so


class Bridge:
    """A context of the library built on the fake runtime."""

    def __init__(self, so):
        self.lib = C.CDLL(so)
        for name, res, args in smoe_amd.SIGNATURES:
            if hasattr(self.lib, name):
                getattr(self.lib, name).restype, getattr(self.lib, name).argtypes = res, args
        self.lib.fake_count.restype, self.lib.fake_count.argtypes = C.c_uint64, [C.c_char_p]
        self.lib.fake_budget.argtypes = [C.c_size_t]
        self.lib.fake_is_live.argtypes = [C.c_uint64]
        self.lib.fake_fail.argtypes = [C.c_char_p]
        self.budget()
        self.capturing(False)
        self.ctx = self.lib.smoe_metal_init(1 << 15)
        assert self.ctx

    def close(self):
        self.capturing(False)
        self.lib.smoe_metal_destroy(self.ctx)
        assert self.count("allocations") == 0 and self.count("host_allocations") == 0   # all given back

    def count(self, what):
        return self.lib.fake_count(what.encode())

    def budget(self, n=None):
        self.lib.fake_budget(C.c_size_t(-1).value if n is None else n)

    def capturing(self, on):
        self.lib.fake_capturing(int(on))

    def live(self, p):
        return bool(self.lib.fake_is_live(p))

    def prefill(self, shape, T, perm=False):
        s = smoe_amd.make_shape(shape["d_model"], shape["n_experts"], shape["top_k"], shape["d_ff"])
        off, _raw, stride = smoe_amd.blob_layout(shape["d_model"], shape["d_ff"])
        layer = smoe_amd.make_layer(DEV, DEV, DEV, stride, off)
        p = DEV if perm else None
        return self.lib.smoe_hip_moe_prefill(self.ctx, C.byref(s), C.byref(layer), DEV, T, None, None, p, p, p, p)

    def group(self, n=2, D=2048, I=768):
        x = np.ones(D, np.float32)
        blobs = (smoe_amd.SmoeExpertBlob * n)(*[smoe_amd.SmoeExpertBlob(*[DEV] * 6, i) for i in range(n)])
        return self.lib.smoe_metal_fused_ffn_group(self.ctx, blobs, n, x.ctypes.data, I, D, D, I, 64, 4)

    def batch(self, n, D=2048, I=768):
        x = np.ones((n, D), np.float32)
        return self.lib.smoe_metal_fused_ffn_batch(self.ctx, *[DEV] * 6, x.ctypes.data, n, I, D, D, I, 64, 4)


@pytest.fixture
def bridge(built):
    b = Bridge(built)
    yield b
    b.close()


@pytest.mark.parametrize("T,dispatches", [(256, 1), (1025, 2), (4096, 2)])
def test_profile_times_every_dispatch_of_a_launcher(bridge, T, dispatches):
    """The permute of several segments takes two dispatches: both are timed, as one launch."""
    L = bridge.lib
    assert L.smoe_hip_profile_enable(bridge.ctx, 1) == 0
    calls = 5000 if T == 1025 else 3     # (past the ring of event slots)
    for _ in range(calls):
        assert bridge.prefill(SHAPE_30B, T) == 0
    n, ms = C.c_uint64(), C.c_double()
    for kind, each in ((smoe_amd.KERNEL_PERMUTE, dispatches), (smoe_amd.KERNEL_ROUTE, 1), (smoe_amd.KERNEL_SCATTER, 1)):
        assert L.smoe_hip_profile_read(bridge.ctx, kind, C.byref(n), C.byref(ms)) == 0
        assert (n.value, ms.value) == (calls, float(calls * each))    # the fake dispatch takes 1 ms
    assert L.smoe_hip_profile_enable(bridge.ctx, 0) == 0


def prefill_bytes(bridge, shape, T):
    """What a context that only runs passes of T tokens of this shape holds for them."""
    before = bridge.count("live")
    assert bridge.prefill(shape, T) == 0
    return bridge.count("live") - before


def test_prefill_scratch_is_what_the_calls_need(built):
    """A long pass of a narrow layer, then a short pass of a wide layer with more experts a token: the
    scratch holds the larger of the two in every buffer, not a long pass of the wide layer, and a
    budget of little more than that is enough."""
    narrow, wide = SHAPE_30B, dict(d_model=8192, n_experts=64, top_k=16, d_ff=4096)
    sizes = []
    for shape, T in ((narrow, 4096), (wide, 16)):
        b = Bridge(built)
        sizes.append(prefill_bytes(b, shape, T))
        b.close()
    b = Bridge(built)
    b.budget(b.count("live") + int(1.1 * sum(sizes)))
    assert b.prefill(narrow, 4096) == 0
    assert b.prefill(wide, 16) == 0
    assert b.prefill(narrow, 4096) == 0 and b.count("T") == 4096
    b.close()


def test_long_pass_that_cannot_be_had_is_not_asked_for_again(built):
    """Where there is memory for passes of 736 tokens only, a longer prompt runs in those: the scratch of
    the calls before stays, and later calls neither allocate nor synchronise."""
    b = Bridge(built)
    short = prefill_bytes(b, SHAPE_30B, 736)
    b.close()
    b = Bridge(built)
    b.budget(b.count("live") + int(1.5 * short))
    assert b.prefill(SHAPE_30B, 736) == 0
    x_hi, frees = b.count("x_hi"), b.count("frees")
    assert b.prefill(SHAPE_30B, 4000) == 0
    assert b.count("failed") > 0 and b.count("T") == 4000 % 736
    assert b.count("x_hi") == x_hi and b.live(x_hi)
    held = b.count("live")
    state = [b.count(w) for w in ("mallocs", "frees", "failed", "syncs")]
    for T in (4000, 4096, 700, 4000):
        assert b.prefill(SHAPE_30B, T) == 0
        assert [b.count(w) for w in ("mallocs", "frees", "failed", "syncs")] == state, T
    assert b.count("x_hi") == x_hi and b.count("live") == held
    # short calls of other shapes that do fit are unaffected
    assert b.prefill(dict(d_model=512, n_experts=8, top_k=2, d_ff=256), 100) == 0 and b.count("T") == 100
    b.close()


def test_captured_prefill_keeps_its_scratch(bridge):
    """A graph holds the scratch it was captured with: a later, longer call grows the scratch beside it.
    Capturing one length after the other, ascending, keeps no more behind than the present scratch."""
    assert bridge.prefill(SHAPE_30B, 1000) == 0
    held = []
    bridge.capturing(True)
    assert bridge.prefill(SHAPE_30B, 512) == 0
    bridge.capturing(False)
    held += [bridge.count("x_hi"), bridge.count("y")]
    assert bridge.prefill(SHAPE_30B, 4000) == 0
    assert bridge.count("x_hi") != held[0] and all(bridge.live(p) for p in held)
    assert bridge.prefill(dict(d_model=4096, n_experts=128, top_k=8, d_ff=1536), 4096) == 0
    assert all(bridge.live(p) for p in held)


def test_ascending_captures_are_bounded(built):
    b = Bridge(built)
    full = prefill_bytes(b, SHAPE_30B, 1024)
    b.close()
    b = Bridge(built)
    base = b.count("live")
    held = []
    for T in range(1, 513):
        assert b.prefill(SHAPE_30B, T) == 0
        b.capturing(True)
        assert b.prefill(SHAPE_30B, T) == 0
        b.capturing(False)
        held.append(b.count("y"))
    assert all(b.live(p) for p in held)
    assert b.count("live") - base <= 2 * full
    b.close()


@pytest.mark.parametrize("shape", [SHAPE_30B, dict(d_model=256, n_experts=8, top_k=2, d_ff=128)])
def test_capture_of_shorter_calls_after_a_longer_one(built, shape):
    """After a call of n tokens, every call of at most n tokens can be captured."""
    for n in (300, 737, 2500, 4096, 4097, 5000, 9000):
        b = Bridge(built)
        assert b.prefill(shape, n) == 0
        b.capturing(True)
        for T in (1, 299, 300, 736, 2049, 2500, 4000, 4096, 4097, 5000, 9000):
            if T <= n:
                assert b.prefill(shape, T) == 0, (n, T)
        b.capturing(False)
        b.close()


@pytest.mark.parametrize("fails,batch", [("gate_up", 0), ("down", 0), ("event_record", 0), ("gate_up_tokens", 9),
                                         ("down_tokens", 9), ("event_record", 9)])
def test_input_copy_of_a_failed_dispatch_is_waited_for(bridge, fails, batch):
    """A dispatch that fails after its input's copy was queued has no handle that says when the copy has read
    the pinned entry: the call waits for it, so that later dispatches may write there."""
    call = (lambda: bridge.batch(batch)) if batch else bridge.group
    assert call()
    dispatches, syncs = bridge.lib.smoe_metal_kernel_dispatches(bridge.ctx), bridge.count("syncs")
    bridge.lib.fake_fail(fails.encode())
    assert call() is None and bridge.count("syncs") == syncs + 1
    if fails != "event_record":
        assert bridge.lib.smoe_metal_kernel_dispatches(bridge.ctx) == dispatches
    for _ in range(8):
        assert call()
    assert bridge.count("syncs") == syncs + 1


def test_longer_batches_find_their_pinned_memory(bridge):
    """The four input entries are as long as the longest dispatch of their kind from their first use on:
    batches that grow by a token allocate no pinned memory of their own."""
    for _ in range(4):
        assert bridge.batch(2) and bridge.group(D=512, I=256)
    n = bridge.count("host_mallocs")
    for k in range(3, 65):
        assert bridge.batch(k) and bridge.group(D=64 * k, I=256)
    assert bridge.count("host_mallocs") == n and bridge.count("host_frees") <= n


def test_permute_outputs_take_the_tokens_that_the_header_states(bridge):
    header = open(os.path.join(ROOT, "include", "smoe_hip.h")).read()
    text = " ".join(header[:header.index("int smoe_hip_moe_prefill(")].replace("*", " ").split())
    limit = int(re.search(r"\((\d+) tokens at 128 experts and top_k 8\); more gives SMOE_ERR_SHAPE", text).group(1))
    assert bridge.prefill(SHAPE_30B, limit, perm=True) == 0 and bridge.count("T") == limit
    assert bridge.prefill(SHAPE_30B, limit + 1, perm=True) == smoe_amd.SMOE_ERR_SHAPE
    assert bridge.prefill(SHAPE_30B, limit + 1) == 0 and bridge.count("T") == limit + 1


@pytest.mark.parametrize("heads,kv_heads,head_dim,wide,plain", [
    # (positions at which k_attn_wide / k_attn_decode measured faster)
    (64, 4, 128, (4096, 8192, 32768), (1, 1000, 3000)),
    (16, 1, 128, (8192, 32768), (4096, 6000)),
    (24, 1, 128, (8192, 10000), (4096, 6000)),
    (40, 1, 128, (4096, 10000), (1000,)),
    (27, 3, 128, (4096, 10000), (1000,)),
    (32, 2, 64, (4096, 8192), (1000,)),
    (16, 1, 64, (4096, 8192), (1000,)),
    (10, 1, 256, (), (2048, 4096, 16384, 32768)),
    (16, 1, 256, (), (4096, 16384, 32768)),
    (24, 1, 256, (8192, 32768), (4096,)),
    (32, 2, 256, (8192, 32768), (4096, 6000)),
    (20, 2, 256, (4096, 6000, 32768), (2048,)),
    (64, 4, 256, (4096, 32768), (1000,)),
    (32, 4, 128, (), (4096, 32768)),
])
def test_attention_takes_the_faster_kernel(built, heads, kv_heads, head_dim, wide, plain):
    f = C.CDLL(built).fake_attn_wide
    assert all(f(heads, kv_heads, head_dim, n) for n in wide)
    assert not any(f(heads, kv_heads, head_dim, n) for n in plain)


@pytest.mark.parametrize("E,K,in_one,in_segments", [
    (128, 8, (257, 300, 512), (64, 256, 640, 736, 4096)),
    (32, 4, (700, 1000), (512, 1500)),
    (8, 2, (1500, 2000), (1000, 4000)),
    (512, 8, (150,), (128, 300)),
])
def test_permute_takes_one_workgroup_where_it_is_faster(bridge, E, K, in_one, in_segments):
    """Batches of several segments that one workgroup holds are permuted by it."""
    shape = dict(d_model=256, n_experts=E, top_k=K, d_ff=128)
    for T in in_one + in_segments:
        one, seg = bridge.count("permutes"), bridge.count("permutes_seg")
        assert bridge.prefill(shape, T) == 0
        got = bridge.count("permutes") - one, bridge.count("permutes_seg") - seg
        assert got == ((1, 0) if T in in_one else (0, 1)), T


def units_of(M, cap):
    """Units of up to cap pairs: (number, of more than 16 rows)."""
    n = -(-M // cap)
    return int(n.sum()), int(n[M > 16].sum())


def shares(lib, n_long, n_short):
    out = (C.c_uint32 * 4)()
    return [(lib.fake_unit_share(x, n_long, n_short, out), tuple(out))[1] for x in range(8)]


def test_work_list_shares(built):
    """Every unit on one XCD, and no XCD with more than an eighth of them rounded up."""
    lib = C.CDLL(built)
    for n_long in range(35):
        for n_short in range(35):
            share = shares(lib, n_long, n_short)
            assert sorted(u for l0, nl, _, _ in share for u in range(l0, l0 + nl)) == list(range(n_long))
            assert sorted(u for _, _, s0, ns in share for u in range(s0, s0 + ns)) == list(range(n_short))
            assert max(nl + ns for _, nl, _, ns in share) == -(-(n_long + n_short) // 8), (n_long, n_short)


def test_work_lists_hold_every_unit(built):
    """Whatever the routing, each XCD's share of the long and of the short units fits the records of the list."""
    lib, rng = C.CDLL(built), np.random.default_rng(3)
    lib.fake_unit_records.restype = C.c_uint64
    for case in range(4000):
        E = int(rng.choice([1, 2, 7, 8, 16, 60, 128, 300, 512]))
        P = int(np.exp(rng.uniform(0, np.log(65536))))
        skew = rng.choice([0.0, 0.5, 1.0, 3.0])
        p = (np.arange(E) + 1.0) ** -skew
        M = rng.multinomial(P, rng.permutation(p) / p.sum())
        if case % 3 == 0:       # as many units as P pairs can make: one pair over a whole number of units
            M = np.zeros(E, np.int64)
            e = min(E, P)
            M[:e] = 1
            left = (P - e) // 32
            for k in range(min(left, 400)):
                M[k % e] += 32
        tiles = int(rng.choice([1, 2, 3, 5, 6, 8, 12, 16, 33, 64]))
        P = int(M.sum())
        u = {cap: units_of(M, cap) for cap in (32, 64)}
        cap = lib.fake_unit_cap(P, u[64][0], u[32][0], tiles)
        slots = lib.fake_unit_slots(P, E, tiles)
        total, long_ = u[cap]
        short = total - long_
        share = shares(lib, long_, short)
        assert max(nl + ns for _, nl, _, ns in share) <= slots // 8, (E, P, tiles, cap)
        assert slots % 8 == 0 and 2 * slots <= lib.fake_unit_records(P, E)


@pytest.mark.parametrize("cap,pairs,u64,u32,tiles", [
    # measured points (kernel us with units of 64 / of 32)
    (32, 514, 16, 23, 10),      # 44.5 / 41.2
    (32, 600, 15, 23, 6),       # 36.7 / 26.8
    (32, 400, 26, 31, 5),       # 22.9 / 17.4
    (32, 600, 15, 23, 4),       # 27.4 / 20.3
    (32, 300, 8, 14, 16),       # 25.9 / 23.3
    (32, 800, 32, 33, 6),       # 32.6 / 29.1
    (32, 512, 57, 62, 6),       # 43.3 / 39.2
    (32, 512, 57, 62, 8),       # 21.1 / 20.6
    (32, 2000, 45, 77, 6),      # 59.1 / 46.0
    (64, 800, 32, 33, 8),       # 15.8 / 22.0
    (64, 514, 16, 23, 12),      # 22.3 / 35.0
    (64, 800, 16, 32, 10),      # 55.7 / 63.5
    (64, 1400, 32, 51, 10),     # 78.7 / 91.8
    (64, 3200, 68, 132, 7),     # 62.4 / 83.4
    (64, 2400, 60, 113, 6),     # 37.7 / 45.3
    (64, 1200, 32, 59, 6),      # 33.4 / 45.0
    (64, 2000, 45, 77, 8),      # 26.3 / 30.6
    (64, 1200, 23, 41, 6),      # 37.2 / 42.3
    (64, 4096, 128, 188, 6),    # 77.0 / 103.5
    (64, 1024, 77, 91, 6),      # 44.2 / 55.0
    (64, 512, 79, 81, 12),      # 130.7 / 143.9
    (64, 2028, 103, 127, 3),    # 22.4 / 25.3
    (64, 704, 16, 24, 11),      # 21.0 / 28.2
])
def test_unit_length_takes_the_faster_cap(built, cap, pairs, u64, u32, tiles):
    assert C.CDLL(built).fake_unit_cap(pairs, u64, u32, tiles) == cap


@pytest.mark.parametrize("pairs,experts,tiles,lds", [
    (128, 16, 10, True), (300, 16, 10, True), (120, 8, 16, True), (16, 1, 6, True), (400, 32, 6, True), (128, 8, 2, True),
    (222, 60, 6, False), (128, 128, 6, False), (900, 60, 5, False), (514, 16, 20, False), (1400, 32, 8, False),
    (4000, 8, 6, False), (4000, 16, 4, False), (8000, 8, 2, False), (1200, 8, 12, False),
])
def test_grouped_launches_of_one_block_a_cu_take_the_lds_kernel(built, pairs, experts, tiles, lds):
    assert bool(C.CDLL(built).fake_lds_weights(pairs, experts, tiles)) == lds
