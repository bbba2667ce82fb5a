"""GPU parity of the prefill attention kernel at the lines between its workgroup shapes: four or eight waves on one query
tile, pairs of tiles from both ends of a causal problem, two groups of waves that share out the keys; with last tiles
that leave whole waves without a query.

Tolerances: a probability is rounded to fp16 once (2^-11 of it), the output once more: at |v| <= 4.5 that is at most
2.2e-3 + 1.1e-3, asked for as 4e-3 + 1e-3 |o|.  Row normalisers 1e-3 + 1e-3 |lse|: the kernel rounds the scaled query to
fp16."""
import pytest
import torch

from oracle import ref

pytestmark = pytest.mark.gpu

N128, N64 = "attn_fwd16_kernel<128, 4, false>", "attn_fwd16_kernel<64, 4, false>"
P128, P64, W128 = "attn_fwd16_kernel<128, 8, true>", "attn_fwd16_kernel<64, 8, true>", "attn_fwd16_kernel<128, 8, false>"
S128, S64 = "attn_fwd16_split_kernel<128>", "attn_fwd16_split_kernel<64>"

# B, Hq, Hkv, Sq, Skv, D, causal, kernel expected
CASES = [
    (4, 32, 8, 270, 270, 128, True, N128), (3, 71, 1, 300, 300, 64, False, N64),          # last tile of 14 / 44 rows: idle waves
    (1, 32, 8, 1430, 1430, 128, True, P128), (1, 32, 8, 1664, 1664, 128, True, P128),     # 12 and 13 tiles: even and odd count
    (2, 16, 4, 1500, 1500, 64, True, P64), (1, 32, 8, 1400, 1400, 128, True, N128),       # ... and 11
    (4, 24, 8, 1000, 1000, 128, True, W128), (4, 24, 8, 900, 900, 128, True, N128),       # 384 tiles of 256: the last nearly full, or not
    (4, 16, 4, 1000, 1000, 128, False, W128), (4, 15, 5, 1000, 1000, 128, False, N128),   # 256 and 240, unmasked
    (1, 16, 2, 1100, 1100, 128, True, S128), (1, 16, 2, 1099, 1099, 128, True, N128),       # the keys' line
    (1, 16, 4, 2060, 2060, 64, True, S64), (2, 16, 4, 1300, 1300, 64, True, N64),         # 272 tiles and 352
    (2, 15, 3, 290, 1225, 128, True, S128), (1, 64, 1, 257, 1216, 64, False, S64),          # fewer queries than keys; odd and even tile counts
    (1, 16, 16, 1152, 1152, 64, False, S64), (1, 32, 8, 300, 1217, 128, False, S128),
]


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,D,causal,name", CASES)
def test_attention_at_the_lines_between_workgroup_shapes(B, Hq, Hkv, Sq, Skv, D, causal, name):
    from triton_amd import ops
    g = torch.Generator().manual_seed(Sq * Skv)
    q, k, v = (ref.randn_half(s, g).cuda() for s in ((B, Hq, Sq, D), (B, Hkv, Skv, D), (B, Hkv, Skv, D)))
    o, lse, scale = torch.full_like(q, 7.0), torch.zeros(B, Hq, Sq, device="cuda"), D ** -0.5
    assert ops.attention_kernel_name(q, k, v, o, scale, causal) == "trn::" + name
    ops.attention(q, k, v, o, scale, causal, lse=lse)
    torch.cuda.synchronize()
    # the reference in float32, a few heads at a time
    keep = None if not causal else torch.ones(Sq, Skv, dtype=torch.bool, device="cuda").tril(Skv - Sq)
    for b in range(B):
        for h in range(Hq):
            s = q[b, h].float() @ k[b, h * Hkv // Hq].float().T * scale
            if causal:
                s = s.masked_fill(~keep, float("-inf"))
            want = s.softmax(-1) @ v[b, h * Hkv // Hq].float()
            err = (o[b, h].float() - want).abs()
            assert not (err > 4e-3 + 1e-3 * want.abs()).any(), f"batch {b} head {h}: max abs err {err.max():.4g}"
            want = torch.logsumexp(s, -1)
            err = (lse[b, h] - want).abs()
            assert not (err > 1e-3 + 1e-3 * want.abs()).any(), f"batch {b} head {h}: max lse err {err.max():.4g}"
