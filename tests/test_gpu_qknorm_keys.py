"""GPU parity of QKNorm attention where the launch normalises the keys itself (scores times the keys' reciprocal root mean squares,
gamma_k in the queries), at the edges of its 32-query and 32-key blocks and in each sharing of the head dimension, and at the line
to the separate launch.  Tolerance: fp16 attention outputs, 2e-2 + 1e-2 |o|."""
import pytest
import torch

from oracle import ref

pytestmark = pytest.mark.gpu


def run(q, k, v, gq, gk, eps, causal=True):
    from triton_amd import modules
    o = torch.full_like(q, 7.0)
    m = modules.get("qknorm", eps=eps, causal=causal)
    t = dict(K=k, O=o, Q=q, V=v, gamma_k=gk, gamma_q=gq)
    m.forward(*[t[p] for p in m.TENSOR_PARAMS])
    torch.cuda.synchronize()
    return o, m


def want(q, k, v, gq, gk, eps, causal=True):
    D, S, G = q.shape[-1], q.shape[2], q.shape[1] // k.shape[1]
    n = lambda x, g: x.double() * (x.double().pow(2).mean(-1, keepdim=True) + eps).rsqrt() * (1 if g is None else g.double())
    s = n(q, gq) @ n(k, gk).repeat_interleave(G, 1).transpose(-1, -2).contiguous() * D ** -0.5
    if causal:
        s = s.masked_fill(~torch.ones(S, S, dtype=torch.bool, device=s.device).tril(), float("-inf"))
    return s.softmax(-1) @ v.double().repeat_interleave(G, 1)


def tensors(B, Hq, Hkv, S, D, seed, std=1.0):
    g = torch.Generator().manual_seed(seed)
    return [ref.randn_half((B, h, S, D), g, 0.0, sd).cuda() for h, sd in ((Hq, 1.0), (Hkv, std), (Hkv, 1.0))] + \
           [ref.randn_half((D,), g, 1.0, 0.1).cuda() for _ in range(2)]


@pytest.mark.parametrize("B,Hq,Hkv,S,D", [(1, 1, 1, 1, 64), (1, 2, 1, 31, 128), (2, 8, 2, 32, 128), (1, 71, 1, 33, 64), (1, 32, 8, 65, 128),
                                          (1, 16, 16, 257, 64), (3, 16, 4, 130, 128), (1, 8, 2, 1000, 128), (7, 71, 1, 20, 64), (1, 1, 1, 2048, 64)])
@pytest.mark.parametrize("weights", [True, False])
def test_keys_normalised_within_the_launch(B, Hq, Hkv, S, D, weights):
    q, k, v, gq, gk = tensors(B, Hq, Hkv, S, D, S + D)
    gq, gk = (gq, gk) if weights else (None, None)
    o, m = run(q, k, v, gq, gk, 1e-5)
    assert len(m._hws) == 0, "no workspace: the keys are not normalised by a launch of their own"
    w = want(q, k, v, gq, gk, 1e-5)
    assert not ((o.double() - w).abs() > 2e-2 + 1e-2 * w.abs()).any()


def test_the_launch_of_its_own_beyond_the_line():
    q, k, v, gq, gk = tensors(1, 1, 1, 2049, 64, 3)
    o, m = run(q, k, v, gq, gk, 1e-5)
    assert len(m._hws) == 1
    w = want(q, k, v, gq, gk, 1e-5)
    assert not ((o.double() - w).abs() > 2e-2 + 1e-2 * w.abs()).any()


@pytest.mark.parametrize("D", [64, 128])
def test_ranges(D):
    """Keys far from unit size, weights whose product leaves fp16, a weight that is zero, a mask-free problem."""
    q, k, v, gq, gk = tensors(1, 4, 2, 70, D, 9, std=200.0)
    k[:, :, ::3] *= 1e-3
    o, _ = run(q, k, v, gq, gk, 1e-5, causal=False)
    w = want(q, k, v, gq, gk, 1e-5, causal=False)
    assert not ((o.double() - w).abs() > 2e-2 + 1e-2 * w.abs()).any()
    ones = torch.ones_like(v)
    o, _ = run(q, k, ones, gq * 300, gk * 300, 1e-5)          # (the winner of such scores hangs on their rounding, the sum does not)
    assert torch.equal(o, torch.ones_like(o))
    o, _ = run(q, k, v, gq, gk * 0, 1e-5)
    w = want(q, k, v, gq, gk * 0, 1e-5)
    assert not ((o.double() - w).abs() > 2e-2 + 1e-2 * w.abs()).any()


# the keys normalised within the attention launch, and by a launch of their own
@pytest.mark.parametrize("B,Hq,S,D", [(2, 8, 100, 128), (2, 71, 300, 64), (3, 40, 515, 128)])
@pytest.mark.parametrize("native", [True, False])
def test_contiguous_keys_of_any_stride_along_an_axis_of_one(B, Hq, S, D, native):
    """A contiguous K may have any stride along an axis of one element: a single KV head seen through the token-major tensor
    that a projection writes, one batch or one key out of a larger buffer."""
    from triton_amd import modules
    g = torch.Generator().manual_seed(S)
    q, k, v = (ref.randn_half((B, h, S, D), g).cuda() for h in (Hq, 1, 1))
    gq, gk = (ref.randn_half((D,), g, 1.0, 0.02).cuda() for _ in range(2))
    m = modules.get("qknorm")

    def out(q, k, v):
        t = dict(Q=q, K=k, V=v, O=torch.full_like(q, 7.0), gamma_q=gq, gamma_k=gk)
        (m.forward if native else m._run)(*[t[p] for p in m.TENSOR_PARAMS])
        torch.cuda.synchronize()
        return t["O"]

    token_major = k.view(B, S, 1, D).transpose(1, 2)
    odd_batch = torch.as_strided(k, (1, 1, S, D), (S * D + 4, 4, D, 1))
    odd_key = torch.as_strided(k, (B, 1, 1, D), (D, 12, 4, 1))
    for odd in (token_major, odd_batch, odd_key):
        b, _, s, _ = odd.shape
        plain = torch.empty(b, 1, s, D, dtype=torch.half, device="cuda").copy_(odd)
        assert odd.is_contiguous() and odd.stride() != plain.stride()
        qs, vs = q[:b, :, :s].contiguous(), v[:b, :, :s].contiguous()
        assert torch.equal(out(qs, odd, vs), out(qs, plain, vs))
