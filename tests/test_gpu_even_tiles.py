"""GPU parity of causal attention whose workgroups take two tiles of 64 queries from the two ends, each with the keys split between
two groups of waves: odd and even tile counts, last tiles that leave waves without a query, the rule's lines.

Tolerance against float64: the scaled queries, the probabilities and the outputs are rounded to fp16 once each, by 2^-11 / sqrt(3) of their
size in root mean square at most: the first shifts a score of standard deviation 1 by 2.8e-4, the three together are 5e-4 in 2-norm.  Row normalisers
1e-3: the scores' shift at |score| <= 4, averaged or not."""
import pytest
import torch

from oracle import ref

pytestmark = pytest.mark.gpu

S128, S64, N128, N64 = "attn_fwd16_split_kernel<128>", "attn_fwd16_split_kernel<64>", "attn_fwd16_kernel<128, 4, false>", "attn_fwd16_kernel<64, 4, false>"
CASES = [
    (1, 12, 4, 1100, 128, S128), (1, 12, 12, 1153, 128, S128), (2, 8, 1, 1216, 128, S128), (1, 28, 4, 1151, 128, S128),      # 18, 19, 19 and 18 tiles; short last ones
    (1, 9, 3, 3583, 128, S128), (1, 2, 2, 8100, 128, S128), (1, 10, 5, 3300, 128, S128),      # 252 workgroups, 128, and 260: one tile
    (1, 14, 7, 600, 64, S64), (1, 14, 7, 599, 64, N64), (3, 14, 14, 705, 64, S64), (2, 20, 4, 769, 64, N64), (1, 16, 2, 1985, 64, S64), (1, 42, 42, 640, 64, S64),
]


@pytest.mark.parametrize("B,Hq,Hkv,S,D,name", CASES)
def test_two_tiles_from_both_ends(B, Hq, Hkv, S, D, name):
    from triton_amd import ops
    g = torch.Generator().manual_seed(S)
    q, k, v = (ref.randn_half((B, h, S, D), g).cuda() for h in (Hq, Hkv, Hkv))
    o, lse = torch.full_like(q, 7.0), torch.zeros(B, Hq, S, device="cuda")
    assert ops.attention_kernel_name(q, k, v, o, D ** -0.5, True) == "trn::" + name
    ops.attention(q, k, v, o, D ** -0.5, True, lse=lse)
    again = torch.zeros_like(o)
    ops.attention(q, k, v, again, D ** -0.5, True)
    assert torch.equal(o, again)
    mask = torch.ones(S, S, dtype=torch.bool, device="cuda").triu(1)
    for b, h in {(0, 0), (B - 1, Hq - 1), (B // 2, Hq // 2)}:
        s = (q[b, h].double() @ k[b, h * Hkv // Hq].double().t() * D ** -0.5).masked_fill_(mask, float("-inf"))
        want = s.softmax(1) @ v[b, h * Hkv // Hq].double()
        rows = (o[b, h] - want).norm(dim=1) / want.norm(dim=1)
        assert (o[b, h] - want).norm() <= 5e-4 * want.norm() and rows.max() <= 2e-3, (rows.max(), rows.argmax())
        assert ((lse[b, h] - s.logsumexp(1)).abs() <= 1e-3).all()


def test_masked_and_large_scores():
    """First keys far below the rest and far above: references that start late in one group of waves, and that have to rise."""
    from triton_amd import ops
    g = torch.Generator().manual_seed(5)
    q, k, v = (ref.randn_half((1, h, 1200, 128), g).cuda() for h in (16, 4, 4))
    q[..., 0] = 8.0
    k[..., 0] = 0.0
    k[:, :, :64, 0], k[:, :, 200:300, 0], k[:, :, 700:, 0] = -100.0, 60.0, -60.0
    o = torch.zeros_like(q)
    ops.attention(q, k, v, o, 128 ** -0.5, True)
    s = (q.double() @ k.double().repeat_interleave(4, 1).transpose(2, 3).contiguous() * 128 ** -0.5)
    s.masked_fill_(torch.ones(1200, 1200, dtype=torch.bool, device="cuda").triu(1), float("-inf"))
    want = s.softmax(-1) @ v.double().repeat_interleave(4, 1)
    # (the keys that count for a row have the same first component, so that the scaled query's rounding there, of scores up to 42, shifts them
    # alike; the rest is as above, twice that for the rows whose few largest scores count)
    assert (o - want).norm() <= 1e-3 * want.norm()
