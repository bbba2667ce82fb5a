"""GPU parity of the decode attention with key statistics over keys split over workgroups (the partial results merged, and the
statistics summed, by a second launch), against fp32 sums and against the single launch.

Tolerances as in test_gpu_scores.py: 2e-2 on outputs of fp16 probabilities, 1e-3 relative on fp32 key scores."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# B, H, Hkv, D, Sq, Skv: as many shares as the rule gives (32 at most; the last one short, of one key, whole) and the least keys
CASES = [(1, 8, 2, 128, 8, 8193), (1, 2, 2, 64, 32, 8192), (1, 16, 16, 64, 5, 2048), (1, 4, 1, 128, 1, 2049), (1, 32, 8, 128, 32, 4112),
         (2, 12, 4, 128, 3, 4097), (1, 71, 71, 64, 16, 4100), (1, 100, 10, 64, 17, 8200), (1, 128, 8, 64, 16, 8192)]


# chunks of more than 32 queries, without noise: the forward's shares
CHUNKS = [(1, 32, 8, 128, 100, 4100), (1, 16, 16, 64, 33, 8193), (1, 71, 1, 64, 128, 9000)]


@pytest.mark.parametrize("B,H,Hkv,D,Sq,Skv", CASES + CHUNKS)
@pytest.mark.parametrize("noise_type", [None, torch.float16, torch.float32])
@pytest.mark.parametrize("causal", [False, True])
def test_shared_out_statistics(B, H, Hkv, D, Sq, Skv, noise_type, causal):
    from triton_amd import ops
    if Sq > 32 and noise_type is not None:
        pytest.skip("chunks are shared out without noise only")
    g = torch.Generator(device="cuda").manual_seed(Skv + Sq)
    q, k, v = (torch.randn(B, h, s, D, generator=g, device="cuda").half() for h, s in ((H, Sq), (Hkv, Skv), (Hkv, Skv)))
    noise = None
    if noise_type is not None:
        noise = (-torch.log(torch.empty(B, H, Sq, Skv, device="cuda").exponential_(generator=g))).to(noise_type)
    scale, tau = D ** -0.5, 1.5 if noise is not None else 1.0
    need = ops.attention_key_scores_workspace_bytes(q, k, v, q, scale, causal, noise is not None)
    assert need > 0
    outs = []
    for ws in (torch.full((need,), 255, dtype=torch.uint8, device="cuda"), None):       # (NaNs to begin with)
        rows, o = torch.zeros(B, H, Sq, device="cuda"), torch.full_like(q, 7.0)
        x, y = torch.full((B, H, Skv), -1.0, device="cuda"), torch.full((B, H, Skv), -1.0, device="cuda")
        ops.attention_key_scores(q, k, v, o, scale, causal, rows, x, y, noise=noise, tau=tau, workspace=ws)
        if ws is not None:
            xh = torch.full((B, H, Skv), -1.0, device="cuda", dtype=torch.float16)
            ops.attention_key_scores(q, k, v, torch.empty_like(q), scale, causal, torch.zeros_like(rows), xh, noise=noise, tau=tau, workspace=ws)
            assert torch.equal(xh, x.half())
        outs.append((o.float(), rows, x, y))
    torch.cuda.synchronize()
    hidden = torch.zeros(Sq, Skv, dtype=torch.bool, device="cuda")
    if causal:
        hidden = ~torch.ones(Sq, Skv, dtype=torch.bool, device="cuda").tril(Skv - Sq)
    for b in range(B):
        kk, vv = (t[b].float().repeat_interleave(H // Hkv, 0) for t in (k, v))
        s = (q[b].float() @ kk.transpose(1, 2).contiguous() * scale).masked_fill(hidden, float("-inf"))
        z = s if noise is None else ((s + noise[b].float().masked_fill(hidden, 0)) / tau)
        p = z.softmax(-1)
        want = s.softmax(-1) @ vv, z.logsumexp(-1), p.sum(1), (p * p).sum(1)
        for o, rows, x, y in outs:
            assert (o[b] - want[0]).abs().max() < 2e-2 and (rows[b] - want[1]).abs().max() < 1e-3
            for got, w in ((x[b], want[2]), (y[b], want[3])):
                assert ((got - w).abs() <= 1e-3 * w + 1e-12).all(), ((got - w).abs() / w).max()


@pytest.mark.parametrize("H,D,noise,keys", [(16, 64, True, 1537), (16, 64, False, 2048), (8, 128, True, 1537), (17, 64, True, 3072), (32, 128, False, 3712),
                                            (64, 128, True, 8192), (128, 64, False, 8192), (129, 64, True, None)])
def test_rule(H, D, noise, keys):
    from triton_amd import ops
    for skv, want in ((16384, keys is not None), (keys, True), ((keys or 1) - 1, False)):
        if skv:
            q, k = torch.empty(1, H, 32, D, dtype=torch.half, device="cuda"), torch.empty(1, 1, skv, D, dtype=torch.half, device="cuda")
            assert (ops.attention_key_scores_workspace_bytes(q, k, k, q, 0.1, True, noise) > 0) == want
            if keys:
                q = torch.empty(1, H, 33, D, dtype=torch.half, device="cuda")
                want = 0 if noise else ops.attention_chunk_workspace_bytes(q, k, k, q, 0.1, True)
                assert ops.attention_key_scores_workspace_bytes(q, k, k, q, 0.1, True, noise) == want
