"""GPU parity of the decode attention with key statistics where the scores stay in registers (at most six key blocks of 32 per
wave, three with the whole head dimension of 128 in one workgroup, two without noise) and one key past it, in every number of column shares.

Tolerances: outputs to 2e-3 of each query's 2-norm (fp16 probabilities and one fp16 rounding, 2^-11 each at most, are some 3e-4 of a
norm; an element of an output is 0.02 to 0.05 at these lengths, so that an absolute bound of that size would see nothing),
1e-3 relative on fp32 key scores as in test_gpu_scores.py."""
import pytest
import torch

from oracle import ref

pytestmark = pytest.mark.gpu

# B, H, Hkv, D, Sq, Skv: four, two and one column shares of 128, two and one of 64; the last kept block full, one key more, one
# block and one key, fewer keys than a block
CASES = [
    (1, 32, 8, 128, 16, 1536), (1, 32, 8, 128, 16, 1537), (1, 8, 2, 128, 32, 1281), (1, 4, 4, 128, 1, 257),
    (2, 50, 10, 128, 5, 1505), (1, 144, 9, 128, 16, 768), (1, 144, 9, 128, 16, 769), (1, 8, 8, 128, 7, 33), (1, 3, 1, 128, 20, 20),
    (1, 71, 71, 64, 16, 1040), (1, 71, 1, 64, 32, 1536), (1, 32, 8, 128, 16, 512), (1, 16, 16, 64, 32, 513), (1, 16, 16, 64, 3, 1537), (1, 150, 15, 64, 16, 1400), (1, 16, 16, 64, 9, 70),
]


@pytest.mark.parametrize("B,H,Hkv,D,Sq,Skv", CASES)
@pytest.mark.parametrize("noise_type", [None, torch.float16, torch.float32])
@pytest.mark.parametrize("causal", [False, True])
def test_kept_scores(B, H, Hkv, D, Sq, Skv, noise_type, causal):
    from triton_amd import ops
    g = torch.Generator().manual_seed(Skv + Sq)
    q, k, v = (ref.randn_half((B, h, s, D), g).cuda() for h, s in ((H, Sq), (Hkv, Skv), (Hkv, Skv)))
    noise = None
    if noise_type is not None:
        gd = torch.Generator(device="cuda").manual_seed(Skv)
        noise = (-torch.log(torch.empty(B, H, Sq, Skv, device="cuda").exponential_(generator=gd))).to(noise_type)
    scale, tau = D ** -0.5, 1.5 if noise is not None else 1.0
    rows, o = torch.zeros(B, H, Sq, device="cuda"), torch.full_like(q, 7.0)
    x, y = torch.full((B, H, Skv), -1.0, device="cuda"), torch.full((B, H, Skv), -1.0, device="cuda")
    ops.attention_key_scores(q, k, v, o, scale, causal, rows, x, y, noise=noise, tau=tau)
    xh = torch.full((B, H, Skv), -1.0, device="cuda", dtype=torch.float16)
    ops.attention_key_scores(q, k, v, torch.empty_like(q), scale, causal, torch.zeros_like(rows), xh, noise=noise, tau=tau)
    torch.cuda.synchronize()
    kk, vv = (t.float().repeat_interleave(H // Hkv, 1) for t in (k, v))
    s = q.float() @ kk.transpose(2, 3).contiguous() * scale
    hidden = torch.zeros(Sq, Skv, dtype=torch.bool, device="cuda")
    if causal:
        hidden = ~torch.ones(Sq, Skv, dtype=torch.bool, device="cuda").tril(Skv - Sq)
    s = s.masked_fill(hidden, float("-inf"))
    want = s.softmax(-1) @ vv
    assert ((o.float() - want).norm(dim=-1) <= 2e-3 * want.norm(dim=-1)).all()
    z = s if noise is None else ((s + noise.float().masked_fill(hidden, 0)) / tau)
    p = z.softmax(-1)
    assert (rows - z.logsumexp(-1)).abs().max() < 1e-3
    for got, want in ((x, p.sum(2)), (y, (p * p).sum(2))):
        assert ((got - want).abs() <= 1e-3 * want + 1e-12).all(), ((got - want).abs() / want).max()
    assert torch.equal(xh, x.half())
