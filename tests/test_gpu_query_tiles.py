"""GPU parity of attention with more than 32 queries per head on both sides of the line between the tiles of 32 queries
(whose eight waves share out the keys) and the prefill kernels.

Tolerances: a probability is rounded to fp16 once (2^-11 of it), the output once more: at |v| <= 4.5 that is at most
2.2e-3 + 1.1e-3, asked for as 4e-3 + 1e-3 |o|.  Row normalisers 1e-3 + 1e-3 |lse|: the prefill kernel rounds the scaled
query to fp16."""
import pytest
import torch

from oracle import ref

pytestmark = pytest.mark.gpu


def close(got, want, atol, rtol):
    err = (got.float().cpu() - want.float()).abs()
    assert not (err > atol + rtol * want.float().abs()).any(), f"max abs err {err.max():.4g}"


# B, Hq, Hkv, Sq, Skv, D, causal, with noise, 32-query tiles expected
CASES = [
    (1, 4, 4, 33, 33, 128, True, False, True), (1, 4, 2, 64, 200, 64, True, False, True),      # tile edges, 4 / 2 column shares
    (1, 9, 3, 65, 1000, 128, False, False, True), (1, 71, 1, 96, 96, 64, True, False, True),   # heads no multiple of 8
    (1, 32, 8, 256, 256, 128, True, False, True), (1, 32, 8, 257, 257, 128, True, False, False),   # 256 tiles and 288
    (2, 16, 16, 230, 230, 64, True, False, True), (2, 16, 16, 260, 260, 64, False, False, False),
    (1, 71, 1, 100, 1024, 64, False, False, True), (1, 71, 1, 100, 1023, 64, False, False, False),   # 284 tiles, long keys or not
    (1, 32, 32, 100, 1500, 128, False, True, True), (1, 71, 71, 70, 333, 64, True, True, True),      # score perturbation
    # a few heads, or a number that is no multiple of 8, with so many tiles that they are spread over the XCDs: 4, 2 and 1 column
    # shares, numbers of tiles that are no multiple of 8, the number of workgroups from which on they are (33 of a head per XCD)
    (1, 1, 1, 1100, 1100, 64, True, False, True), (1, 3, 1, 530, 530, 128, False, False, True), (1, 12, 4, 300, 300, 128, True, True, True),
    (3, 3, 3, 800, 830, 64, True, False, True), (1, 1, 1, 512, 600, 64, False, False, True), (1, 1, 1, 513, 600, 64, False, True, True),
    (1, 32, 8, 480, 480, 128, True, True, True), (1, 32, 8, 500, 520, 128, True, True, False),       # 480 tiles and 512
]


# few heads of 128 under a causal mask: past a tile a CU
FEW = [
    (1, 4, 1, 3584, 3584, 128, True, False, True), (1, 4, 1, 3585, 3585, 128, True, False, False), (1, 8, 2, 1025, 1025, 128, True, False, True),
    (1, 8, 2, 1600, 1600, 128, True, False, True), (1, 8, 2, 1601, 1601, 128, True, False, False), (1, 8, 2, 1200, 1201, 128, True, False, False),
    (1, 8, 8, 1100, 1100, 128, False, False, False), (2, 5, 5, 1117, 1117, 128, True, False, True), (1, 10, 2, 1121, 1121, 128, True, False, False),
    (1, 12, 4, 861, 861, 128, True, False, True), (1, 12, 4, 865, 865, 128, True, False, False), (1, 13, 1, 700, 700, 128, True, False, False),
]


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,D,causal,with_noise,tiles", CASES + FEW)
def test_attention_on_both_sides_of_the_query_tile_rule(B, Hq, Hkv, Sq, Skv, D, causal, with_noise, tiles):
    from triton_amd import ops
    g = torch.Generator().manual_seed(Sq * Skv)
    q, k, v = (ref.randn_half(s, g) for s in ((B, Hq, Sq, D), (B, Hkv, Skv, D), (B, Hkv, Skv, D)))
    scale, tau = D ** -0.5, 1.5
    qd, kd, vd = q.cuda(), k.cuda(), v.cuda()
    o, lse = torch.full_like(qd, 7.0), torch.zeros(B, Hq, Sq, device="cuda")
    kw = {}
    if with_noise:
        noise = ref.gumbel_noise((B, Hq, Sq, Skv), 5)
        buf = torch.full((B, Hq, Sq, (Skv + 3) // 4 * 4), float("nan"), device="cuda")
        buf[..., :Skv] = noise.cuda()
        kw = dict(noise=buf[..., :Skv], tau=tau, lse_pert=torch.zeros(B, Hq, Sq, device="cuda"))
    assert ("attn_decode_kernel" in ops.attention_kernel_name(qd, kd, vd, o, scale, causal, with_noise)) == tiles
    ops.attention(qd, kd, vd, o, scale, causal, lse=lse, **kw)
    torch.cuda.synchronize()
    want, want_lse = ref.attention(q, k, v, scale, causal, return_lse=True)
    close(o, want, 4e-3, 1e-3)
    close(lse, want_lse, 1e-3, 1e-3)
    if with_noise:
        z = (ref.scores_fp32(q, k, scale, causal) + noise) / tau
        close(kw["lse_pert"], torch.logsumexp(z, -1), 1e-3, 1e-3)
