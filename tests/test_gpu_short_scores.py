"""GPU parity of attention with key statistics in one launch on short prompts (33 to 128 queries, at most 128 keys) and one past.

Tolerances: outputs to 2e-3 of each query's 2-norm (fp16 probabilities and one fp16 rounding, 2^-11 each at most, are some 3e-4
of a norm), 1e-3 relative on fp32 key scores as in test_gpu_scores.py; a deviation is known to 1e-3 of its column's root mean square."""
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [(1, 4, 4, 128, 33, 33), (1, 6, 2, 64, 64, 64), (2, 8, 2, 128, 65, 65), (6, 16, 16, 64, 100, 100), (1, 32, 8, 128, 128, 128),
         (1, 71, 1, 64, 128, 128), (2, 3, 3, 128, 33, 128), (1, 5, 1, 64, 97, 127), (1, 4, 2, 128, 129, 129), (1, 4, 2, 64, 128, 129)]


@pytest.mark.parametrize("B,H,Hkv,D,Sq,Skv", CASES)
@pytest.mark.parametrize("noise_type", [None, torch.float16, torch.float32])
@pytest.mark.parametrize("causal", [False, True])
def test_short_prompts(B, H, Hkv, D, Sq, Skv, noise_type, causal):
    from triton_amd import ops
    g = torch.Generator(device="cuda").manual_seed(Skv + Sq)
    q, k, v = (torch.randn(B, h, s, D, generator=g, device="cuda").half() for h, s in ((H, Sq), (Hkv, Skv), (Hkv, Skv)))
    noise, tau, scale = None, 1.0, D ** -0.5
    hidden = torch.zeros(Sq, Skv, dtype=torch.bool, device="cuda")
    if causal:
        hidden = ~torch.ones(Sq, Skv, dtype=torch.bool, device="cuda").tril(Skv - Sq)
    if noise_type is not None:          # rows that begin on an odd element; what no query sees is NaN
        tau = 1.5
        store = torch.full((B * H * Sq * (Skv + 1) + 1,), float("nan"), dtype=noise_type, device="cuda")
        noise = torch.as_strided(store, (B, H, Sq, Skv), (H * Sq * (Skv + 1), Sq * (Skv + 1), Skv + 1, 1), 1)
        noise.copy_((-torch.log(torch.empty(B, H, Sq, Skv, device="cuda").exponential_(generator=g))).masked_fill(hidden, float("nan")))

    def run(dtype, two, mean_std):
        rows, o = torch.zeros(B, H, Sq, device="cuda"), torch.full_like(q, 7.0)
        x, y = (torch.full((B, H, Skv), -1.0, device="cuda", dtype=dtype) for _ in range(2))
        ops.attention_key_scores(q, k, v, o, scale, causal, rows, x, y if two else None, noise=noise, tau=tau, mean_std=mean_std)
        torch.cuda.synchronize()
        return o, rows, x, y
    o, rows, x, y = run(torch.float32, True, False)
    half = run(torch.float16, False, False)
    assert torch.equal(half[0], o) and torch.equal(half[1], rows) and torch.equal(half[2], x.half()) and (half[3] == -1).all()
    kk, vv = (t.double().repeat_interleave(H // Hkv, 1) for t in (k, v))
    s = (q.double() @ kk.transpose(2, 3).contiguous() * scale).masked_fill(hidden, float("-inf"))
    want = s.softmax(-1) @ vv
    assert ((o.double() - want).norm(dim=-1) <= 2e-3 * want.norm(dim=-1)).all()
    z = s if noise is None else ((s + noise.double()) / tau).masked_fill(hidden, float("-inf"))
    p = z.softmax(-1)
    assert (rows - z.logsumexp(-1)).abs().max() < 1e-3
    for got, want in ((x, p.sum(2)), (y, (p * p).sum(2))):
        assert ((got - want).abs() <= 1e-3 * want + 1e-12).all(), ((got - want).abs() / want).max()
    if noise is None:
        o2, rows2, mean, std = run(torch.float32, True, True)
        n = (~hidden).sum(0).double()
        m1, m2 = p.sum(2) / n, (p * p).sum(2) / n
        assert torch.equal(o, o2) and torch.equal(rows, rows2)
        assert ((mean - m1).abs() <= 1e-3 * m1).all() and ((std - (m2 - m1 * m1).clamp(min=0).sqrt()).abs() <= 1e-3 * m2.sqrt()).all()
