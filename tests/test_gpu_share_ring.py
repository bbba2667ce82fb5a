"""A chunk of queries on a long cache, its keys shared out: shares of every small number of 64-key tiles (one group of waves has one
fewer, or none), last shares that are short or empty, a last block that is partly past the keys, rings longer and shorter than a
walk, the causal diagonal in every place of the ring.  Against the float64 softmax.

Tolerances as in test_gpu_key_shares.py.  With `shift` every score lies some 110 (nat) below zero, so that whatever a stage without
keys would give (zeros: a score of 0) must not become a reference: the weights of the real keys would be 2^-160, i.e. nothing.  The
scaled queries are rounded to fp16, 2^-11 of each product, which moves a row's normaliser by up to 2^-11 of the scores' size, and
the weights by the spread of the keys around their mean only."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# heads of 128 queries -> min(16, 256 / heads) shares
@pytest.mark.parametrize("H,Hkv,Sq,Skv,D", [
    (1, 1, 40, 3072, 128), (2, 1, 33, 3137, 128), (3, 3, 128, 4097, 128),     # 3, 4 and 5 tiles, 16 shares: 16, 13 and 13 with keys
    (20, 4, 100, 3201, 128), (32, 8, 70, 3105, 128), (64, 64, 35, 3073, 128), (128, 8, 50, 3071 + 65, 128),    # 12, 8, 4 and 2 shares
    (1, 1, 40, 4096, 64), (16, 2, 60, 5060, 64), (71, 1, 128, 2561, 64), (128, 128, 33, 4159, 64), (100, 10, 97, 4129, 64)])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("shift", [0.0, 10.0])
def test_share_walks(H, Hkv, Sq, Skv, D, causal, shift):
    from triton_amd import ops
    g = torch.Generator(device="cuda").manual_seed(Skv + H)
    r = lambda h, s: torch.randn(1, h, s, D, generator=g, device="cuda")
    q, k, v = r(H, Sq), r(Hkv, Skv), r(Hkv, Skv).half()
    scale = D ** -0.5
    if shift:
        q, k = 1 + 0.1 * q, k - shift * (128 / D) ** 0.5
    q, k = q.half(), k.half()
    o, lse = torch.full_like(q, 7.0), torch.zeros(1, H, Sq, device="cuda")
    n = ops.attention_chunk_workspace_bytes(q, k, v, o, scale, causal)
    assert n > 0
    ops.attention(q, k, v, o, scale, causal, lse=lse, workspace=torch.full((n,), 0xFF, dtype=torch.uint8, device="cuda"))
    torch.cuda.synchronize()
    for h in range(H):
        s = q[0, h].double() @ k[0, h // (H // Hkv)].double().T * scale
        if causal:
            s = s.masked_fill(~torch.ones(Sq, Skv, dtype=torch.bool, device="cuda").tril(Skv - Sq), float("-inf"))
        want, rows = s.softmax(-1) @ v[0, h // (H // Hkv)].double(), s.logsumexp(-1)
        assert ((o[0, h].double() - want).abs() <= 4e-3 + 1e-3 * want.abs()).all(), h
        assert ((lse[0, h].double() - rows).abs() <= 2e-3 + 2.0 ** -11 * rows.abs()).all(), h
