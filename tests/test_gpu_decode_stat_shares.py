"""GPU parity of the decode attention with key statistics over keys split over workgroups (the partial results merged, and the
statistics summed, by a second launch), against fp32 sums and against the single launch.

Tolerances: outputs to 2e-3 of each query's 2-norm (fp16 probabilities and one fp16 rounding, 2^-11 each at most, are some 3e-4 of a
norm; an element of an output is 0.02 to 0.05 at these lengths, so that an absolute bound of that size would see nothing),
1e-3 relative on fp32 key scores as in test_gpu_scores.py."""
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
            assert ((o[b] - want[0]).norm(dim=-1) <= 2e-3 * want[0].norm(dim=-1)).all() and (rows[b] - want[1]).abs().max() < 1e-3
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


# the shares by the statistics' rule, by that of the plain attention's workspace too (4112 keys, 16 heads), and none of either
@pytest.mark.parametrize("B,H,Hkv,D,Sq,Skv", [(1, 8, 8, 128, 8, 4112), (1, 16, 16, 64, 5, 4112), (1, 8, 2, 128, 32, 8193), (1, 100, 10, 64, 17, 9000),
                                              (1, 2, 1, 64, 1, 2049), (1, 8, 8, 128, 8, 700),
                                              (1, 32, 32, 128, 3, 3800), (1, 5, 5, 64, 9, 7001)])        # six shares of eight, sixteen of 32
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("half", [False, True])
def test_mean_and_deviation_of_shared_out_keys(B, H, Hkv, D, Sq, Skv, causal, half):
    """At most 32 queries, mean and standard deviation, a workspace of any contents: against float64.

    Bounds: the normaliser sums probabilities rounded to fp16 (2^-12 relative at most, each), hence 2.5e-4 on the means; a
    difference of the two sums that is known to 1e-7 of E p^2 gives its root to 3e-4 of the root mean square; fp16 results
    are rounded once more (2^-11, and half of the smallest fp16 number)."""
    from triton_amd import ops
    g = torch.Generator(device="cuda").manual_seed(Skv + Sq)
    q, k, v = (torch.randn(B, h, s, D, generator=g, device="cuda").half() for h, s in ((H, Sq), (Hkv, Skv), (Hkv, Skv)))
    scale = D ** -0.5
    size = max(ops.attention_key_scores_workspace_bytes(q, k, v, q, scale, causal, False), ops.attention_workspace_bytes(q, k, v, q, scale, causal))
    ws = torch.full((max(size, 256),), 255, dtype=torch.uint8, device="cuda")
    rows, o = torch.full((B, H, Sq), -1.0, device="cuda"), torch.full_like(q, 7.0)
    out = [torch.full((B, H, Skv), -1.0, device="cuda", dtype=torch.half if half else torch.float) for _ in range(2)]
    ops.attention_key_scores(q, k, v, o, scale, causal, rows, *out, mean_std=True, workspace=ws)
    torch.cuda.synchronize()
    seen = torch.ones(Sq, Skv, dtype=torch.bool, device="cuda")
    if causal:
        seen = seen.tril(Skv - Sq)
    n = seen.sum(0).double()
    rounded, least = (2.0 ** -11, 2.0 ** -25) if half else (0.0, 0.0)
    for h in range(H):
        kk, vv = (t[0, h * Hkv // H].double() for t in (k, v))
        s = (q[0, h].double() @ kk.T.contiguous() * scale).masked_fill(~seen, float("-inf"))
        p = s.softmax(-1)
        want = p @ vv
        assert ((o[0, h].double() - want).norm(dim=-1) <= 2e-3 * want.norm(dim=-1)).all() and (rows[0, h].double() - s.logsumexp(-1)).abs().max() <= 2.5e-4
        mean, square = p.sum(0) / n, p.pow(2).sum(0) / n
        std = (square - mean * mean).clamp(min=0).sqrt()
        std[n == 1] = 0
        assert ((out[0][0, h].double() - mean).abs() <= (2.5e-4 + rounded) * mean + least).all()
        assert ((out[1][0, h].double() - std).abs() <= 2.5e-4 * std + 3e-4 * square.sqrt() + rounded * std + least).all()


# problems that use no workspace, that use one, that share out a chunk's keys, and prompts with two launches
@pytest.mark.parametrize("B,H,Hkv,D,Sq,Skv", [(1, 8, 8, 128, 8, 200), (1, 8, 8, 128, 8, 4112), (1, 16, 16, 64, 5, 2064), (1, 8, 8, 128, 100, 4100),
                                              (1, 4, 2, 64, 300, 300), (1, 4, 2, 128, 64, 64)])
@pytest.mark.parametrize("mean_std", [False, True])
def test_a_misaligned_workspace_is_not_used(B, H, Hkv, D, Sq, Skv, mean_std):
    """Off 256 bytes: the call is the one without a workspace, and nothing is written there."""
    from triton_amd import ops
    g = torch.Generator(device="cuda").manual_seed(Skv)
    q, k, v = (torch.randn(B, h, s, D, generator=g, device="cuda").half() for h, s in ((H, Sq), (Hkv, Skv), (Hkv, Skv)))
    assert ops.attention_stats_workspace_bytes(q, k, v, q, D ** -0.5, True) == 0
    need = max(256, ops.attention_key_scores_workspace_bytes(q, k, v, q, D ** -0.5, True, False), ops.attention_workspace_bytes(q, k, v, q, D ** -0.5, True))
    store = torch.full((need + 16,), 255, dtype=torch.uint8, device="cuda")
    assert store.data_ptr() % 256 == 0
    results = []
    for ws in (None, store[16:]):
        rows, o = torch.zeros(B, H, Sq, device="cuda"), torch.full_like(q, 7.0)
        x, y = (torch.full((B, H, Skv), -1.0, device="cuda") for _ in range(2))
        ops.attention_key_scores(q, k, v, o, D ** -0.5, True, rows, x, y, mean_std=mean_std, workspace=ws)
        results.append((o, rows, x, y))
    torch.cuda.synchronize()
    assert (store == 255).all()
    for a, b in zip(*results):
        assert torch.equal(a, b)


def test_a_misaligned_workspace_is_refused_where_it_was():
    """The sizes and problems of attention_stats_workspace_bytes."""
    from triton_amd import ops
    q, k = torch.zeros(1, 8, 8, 128, dtype=torch.half, device="cuda"), torch.zeros(1, 8, 8192, 128, dtype=torch.half, device="cuda")
    need = ops.attention_stats_workspace_bytes(q, k, k, q, 0.1, True)
    assert need > 0
    rows, x = torch.zeros(1, 8, 8, device="cuda"), torch.zeros(1, 8, 8192, device="cuda")
    with pytest.raises(Exception, match="ALIGN"):
        ops.attention_key_scores(q, k, k, torch.empty_like(q), 0.1, True, rows, x, workspace=torch.zeros(need + 16, dtype=torch.uint8, device="cuda")[16:])


@pytest.mark.parametrize("general", [False, True])
@pytest.mark.parametrize("B,H,Hkv,D,Sq,Skv", CASES[:4] + [(1, 16, 16, 64, 20, 2100)])
def test_the_keyformer_module_shares_out_the_keys_of_few_queries(B, H, Hkv, D, Sq, Skv, general):
    """A few queries on a long cache through the module: split over workgroups as by the call that is given a workspace -- the same
    bits -- with one of its own.  general: scores that the kernels do not write themselves (the path in Python)."""
    from triton_amd import modules, ops
    g = torch.Generator(device="cuda").manual_seed(Skv + Sq)
    q, k, v = (torch.randn(B, h, s, D, generator=g, device="cuda").half() for h, s in ((H, Sq), (Hkv, Skv), (Hkv, Skv)))
    noise = -torch.log(torch.empty(B, H, Sq, Skv, device="cuda").exponential_(generator=g))
    c = torch.empty(B, H, 2 * Skv, device="cuda")[..., ::2] if general else torch.empty(B, H, Skv, device="cuda")
    m, o = modules.get("keyformer", tau=1.5), torch.empty_like(q)
    t = dict(Q=q, K=k, V=v, O=o, noise=noise, C_out=c)
    m.forward(*[t[p] for p in m.TENSOR_PARAMS])
    outs = []
    need = ops.attention_key_scores_workspace_bytes(q, k, v, o, D ** -0.5, True, True)
    for ws in (torch.empty(need, dtype=torch.uint8, device="cuda"), None):
        rows, x, ow = torch.empty(B, H, Sq, device="cuda"), torch.empty(B, H, Skv, device="cuda"), torch.empty_like(q)
        ops.attention_key_scores(q, k, v, ow, D ** -0.5, True, rows, x, noise=noise, tau=1.5, workspace=ws)
        outs.append((ow, x))
    torch.cuda.synchronize()
    assert torch.equal(o, outs[0][0]) and torch.equal(c, outs[0][1]) and any(key[0] == "key_parts" for key in m._ws)
    assert (c - outs[1][1]).abs().max() <= 1e-4 * c.abs().max()


# 24 shares and the 16 below that line, eight of head_dim 64, twelve on a longer cache
@pytest.mark.parametrize("B,H,Hkv,D,Sq,Skv", [(1, 8, 2, 128, 3, 11000), (1, 10, 10, 64, 32, 10999), (1, 3, 1, 128, 2, 9001), (1, 26, 26, 64, 5, 8200), (1, 17, 17, 64, 1, 10000)])
@pytest.mark.parametrize("noise_type", [None, torch.float16])
def test_numbers_of_shares(B, H, Hkv, D, Sq, Skv, noise_type):
    test_shared_out_statistics(B, H, Hkv, D, Sq, Skv, noise_type, True)
