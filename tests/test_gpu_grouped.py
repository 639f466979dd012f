"""The grouped prefill GEMMs and the segmented permute at the edges of their
units: work lists of units of up to 32 pairs (few blocks) and of up to 64
(test_units_of_48_and_64_rows), long units before short ones, pair counts around
every 16-row tile, rows of one to several pairs of 64-column groups (with and
without a remainder), small grids and odd numbers of groups (the LDS-weight kernel)
and larger grids (the register kernel: more than 256 experts with a pair, or
several row tiles), batches over several permute segments and over one pass.  Every result against fp64
(moe_delta_f64_batch) and bit for bit against the same tokens in calls of 16."""
import numpy as np
import pytest
import torch

from gpu_helpers import Layer, hidden_states, moe_delta_f64_batch, rel_err

pytestmark = pytest.mark.gpu
TOL_F64 = 5e-4   # of test_gpu_prefill's comparison with fp64


def prefill(ctx, layer, h, step):
    out = h.clone()
    T, K = h.shape[0], layer.K
    ids = torch.zeros((T, K), dtype=torch.int32, device="cuda")
    w = torch.zeros((T, K), dtype=torch.float32, device="cuda")
    for t in range(0, T, step):
        n = min(step, T - t)
        ctx.moe_prefill(layer.shape, layer.layer, out[t].data_ptr(), n, ids[t].data_ptr(), w[t].data_ptr())
    ctx.synchronize()
    return out, ids, w


@pytest.mark.parametrize("D,E,K,I,Ts", [
    (384, 1, 1, 128, (1, 15, 16, 17, 32, 33, 48, 49, 63, 64, 65, 97, 129, 200)),   # every pair on one expert
    (128, 1, 1, 640, (16, 33, 65)),      # one pair of groups in, five out
    (1280, 4, 2, 704, (37, 150)),        # an odd number of groups in the down rows
    (320, 8, 3, 192, (50,)),             # and in both
    (1152, 4, 2, 896, (9, 70)),          # odd numbers of pairs of groups past the first ring of stages
    (256, 512, 8, 128, (300,)),          # segments of 16 chunks
    (256, 128, 8, 128, (257, 1000, 5000)),   # several segments, several passes
    (128, 300, 4, 128, (290, 1100, 2400)),   # more than a block a CU: the register kernel, one stage
    (384, 260, 4, 256, (1000, 2600)),        # three stages of gate/up, two of down
    (640, 260, 2, 640, (3800,)),             # five of both
])
def test_passes_and_segments(ctx, D, E, K, I, Ts):
    check(ctx, D, E, K, I, Ts)


def check(ctx, D, E, K, I, Ts):
    """The ids of every call."""
    layer = Layer(ctx, D, E, K, I, layer_id=500 + D + I)
    all_ids = []
    hs = hidden_states(ctx, min(max(Ts), 512), D, index0=77)
    hs = hs.repeat((max(Ts) + len(hs) - 1) // len(hs), 1)
    hs[:, 0] += torch.arange(len(hs), device="cuda") * 1e-3      # (repeated rows differ)
    for T in Ts:
        print(f"case D={D} E={E} K={K} I={I} T={T}", flush=True)
        h = hs[:T].contiguous()
        out, ids, w = prefill(ctx, layer, h, T)
        out16, ids16, w16 = prefill(ctx, layer, h, 16)
        assert torch.equal(ids, ids16) and torch.equal(w, w16) and torch.equal(out, out16)
        rows = np.unique(np.linspace(0, T - 1, 200).astype(int))
        x = h.cpu().numpy()[rows]
        ref = moe_delta_f64_batch(layer, x, ids.cpu().numpy()[rows], w.cpu().numpy()[rows])
        got = out.cpu().numpy()[rows]
        err, _ = rel_err(got.astype(np.float64) - x, ref, slack=np.spacing(np.abs(got)))
        assert err <= TOL_F64, f"T={T}: {err:.2e}"
        all_ids.append(ids.cpu().numpy())
    return all_ids


def unit_rows(ids, E, tiles):
    """Rows of the units of the work list that the permute of ids makes for a launch of so many row tiles: an
    expert's M pairs in units of up to 32 or 64 (unit_cap), in equal numbers of 16-row tiles."""
    M = np.bincount(ids.ravel(), minlength=E)
    u64, u32 = np.sum(-(-M // 64)), np.sum(-(-M // 32))
    b64, b32 = -(-u64 // 8) * tiles, -(-u32 // 8) * tiles
    small = b32 <= 32 or (b64 > 32 and b32 <= 64 and (8 * u32 <= 9 * u64 or M.sum() >= 40 * u64))
    cap = 32 if small else 64
    n, m16 = -(-M // cap), -(-M // 16)
    return {16 * -(-int(t) // int(k)) for t, k in zip(m16, n) if k}


@pytest.mark.parametrize("D,E,K,I,Ts", [
    (256, 32, 4, 2048, (300, 450, 640)),     # two stages of gate/up
    (1152, 36, 4, 1920, (380, 560)),         # odd numbers of stages, also of down
    (128, 64, 4, 1152, (660, 900)),          # one stage of gate/up
    (128, 300, 4, 128, (2900, 3900)),        # one stage of both
    (1600, 32, 4, 2112, (300, 450, 640)),    # odd numbers of groups: the LDS-weight kernel
])
def test_units_of_48_and_64_rows(ctx, D, E, K, I, Ts):
    """Wide layers with enough experts for units of up to 64 pairs: the 48- and the 64-row forms of both
    kernels give every pair the sums of the 16-row form."""
    seen = [set(), set()]
    for ids in check(ctx, D, E, K, I, Ts):
        for s, tiles in zip(seen, (-(-I // 128), -(-D // 256))):
            s |= unit_rows(ids, E, tiles)
    assert {48, 64} <= seen[0], seen
    assert {48, 64} <= seen[1] or -(-D // 256) == 1 and E < 300, seen
