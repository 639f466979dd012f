"""Device-resident decode MoE block (smoe_hip_moe_decode) against the CPU
oracle of decode.cpp:236-509.  Top-k ids must be bit-exact; the MoE delta and
the post-residual hidden state within 1e-3 per element (rel_err metric)."""
import numpy as np
import pytest
import torch

from gpu_helpers import Layer, hidden_states, moe_delta_err, rel_err

pytestmark = pytest.mark.gpu
TOL = 1e-3


def run_and_check(ctx, oracle, layer, T=1, index0=0):
    hid = hidden_states(ctx, T, layer.D, index0)
    h0 = hid.cpu().numpy()
    ids = torch.zeros((T, layer.K), dtype=torch.int32, device="cuda")
    w = torch.zeros((T, layer.K), dtype=torch.float32, device="cuda")
    ctx.moe_decode(layer.shape, layer.layer, hid.data_ptr(), T, ids.data_ptr(), w.data_ptr())
    torch.cuda.synchronize()
    got = hid.cpu().numpy()
    gids = ids.cpu().numpy().view(np.uint32)
    gw = w.cpu().numpy()
    worst = 0.0
    for t in range(T):
        out, oid, ow, logits, normed, yo = layer.oracle_decode(oracle, h0[t])
        assert (gids[t] == oid).all(), (t, gids[t], oid)
        assert np.allclose(gw[t], ow, rtol=1e-5, atol=1e-7)
        e1, _ = moe_delta_err(got[t], h0[t], yo, ow)
        e2, _ = rel_err(got[t], out)
        worst = max(worst, e1, e2)
        # routing margin between rank k-1 and rank k (reported, not asserted)
        p = np.exp(logits - logits.max())
        p /= p.sum()
        srt = np.sort(p)[::-1]
        print(f"t={t} rel_err delta={e1:.2e} hidden={e2:.2e} margin_k={srt[layer.K - 1] - srt[layer.K]:.3e}")
    assert worst <= TOL, worst
    return worst


def test_tiny_shapes(ctx, oracle):
    for (D, E, K, I) in ((64, 8, 2, 64), (128, 16, 4, 192), (256, 64, 8, 128), (512, 200, 6, 256)):
        layer = Layer(ctx, D, E, K, I, layer_id=D + E)
        run_and_check(ctx, oracle, layer, T=2)


def test_qwen3_30b_layer(ctx, oracle):
    """Config 1: one Qwen3-30B-A3B-shaped layer, batch-1 decode."""
    layer = Layer(ctx, 2048, 128, 8, 768)
    run_and_check(ctx, oracle, layer, T=1)
    run_and_check(ctx, oracle, layer, T=3, index0=10)


def test_qwen3_235b_layer(ctx, oracle):
    """Config 3 shape: one Qwen3-235B-A22B-shaped layer."""
    layer = Layer(ctx, 4096, 128, 8, 1536, layer_id=7)
    run_and_check(ctx, oracle, layer, T=1)


def test_no_renorm_and_k16(ctx, oracle):
    layer = Layer(ctx, 512, 128, 16, 256, layer_id=3, norm_topk=False)
    run_and_check(ctx, oracle, layer, T=2)


def test_graph_replay_matches_eager(ctx, oracle):
    """Two layers captured in a HIP graph and replayed: every replay equals the
    eager result (no memset nodes; the route counter is reset by the kernel)."""
    l0 = Layer(ctx, 2048, 128, 8, 768, layer_id=0, host=False)
    l1 = Layer(ctx, 2048, 128, 8, 768, layer_id=1, host=False)
    x0 = hidden_states(ctx, 1, 2048, 77)
    eager = x0.clone()
    ctx.moe_decode(l0.shape, l0.layer, eager.data_ptr(), 1)
    ctx.moe_decode(l1.shape, l1.layer, eager.data_ptr(), 1)
    torch.cuda.synchronize()
    buf = x0.clone()
    s = torch.cuda.Stream()
    ctx.reserve(l0.shape, 1)
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        ctx.set_stream(s.cuda_stream)
        with torch.cuda.graph(g, stream=s):
            ctx.moe_decode(l0.shape, l0.layer, buf.data_ptr(), 1)
            ctx.moe_decode(l1.shape, l1.layer, buf.data_ptr(), 1)
    ctx.set_stream(torch.cuda.current_stream().cuda_stream)
    for _ in range(4):
        buf.copy_(x0)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(buf, eager)


@pytest.mark.parametrize("D,E,K,I,Ts", [
    (2048, 128, 8, 768, (2, 5, 11, 24)),    # two, two, five and ten row blocks a wave
    (512, 16, 4, 256, (2, 7)),              # one row block a wave
    (4096, 128, 8, 1536, (5,)),             # two chunks a lane: rows loaded block by block
    (1280, 60, 6, 704, (11, 40)),           # an odd number of row blocks
    (512, 200, 6, 256, (90,)),              # more than 128 experts
])
def test_batch_equals_single_calls(ctx, D, E, K, I, Ts):
    """Each token of a batch equals its own two-launch call bit for bit,
    however many row blocks a wave of the batch takes."""
    import smoe_amd
    layer = Layer(ctx, D, E, K, I, layer_id=D + I + 5, host=False)
    for T in Ts:
        print(f"case D={D} E={E} K={K} I={I} T={T}", flush=True)
        x = hidden_states(ctx, T, D, 300)
        batch, one = x.clone(), x.clone()
        ids = torch.zeros((2, T, K), dtype=torch.int32, device="cuda")
        w = torch.zeros((2, T, K), dtype=torch.float32, device="cuda")
        ctx.moe_decode(layer.shape, layer.layer, batch.data_ptr(), T, ids[0].data_ptr(), w[0].data_ptr())
        ctx.set_decode_engine(smoe_amd.DECODE_SPLIT)
        try:
            for t in range(T):
                ctx.moe_decode(layer.shape, layer.layer, one[t].data_ptr(), 1, ids[1, t].data_ptr(), w[1, t].data_ptr())
        finally:
            ctx.set_decode_engine(smoe_amd.DECODE_CHAIN)
        ctx.synchronize()
        assert torch.equal(ids[0], ids[1]) and torch.equal(w[0], w[1])
        assert torch.equal(batch, one) and not torch.equal(batch, x)
