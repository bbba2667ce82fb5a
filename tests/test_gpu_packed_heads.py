"""GPU parity of causal attention whose workgroups take several heads of a KV head: groups that fill them and groups that leave waves
idle, tiles of 32 and 64 queries, short last ones, norms of Q and K, KeyFormer's forward beside the single pass.

Tolerance against float64: the scaled queries, the probabilities and the outputs are rounded to fp16 once each, by 2^-11 / sqrt(3) of their
size in root mean square at most: the first shifts a score of standard deviation 1 by 2.8e-4, the three together are 5e-4 in 2-norm."""
import pytest
import torch

from oracle import ref

pytestmark = pytest.mark.gpu


def compare(q, k, v, o, lse=None):
    B, H, S, D = q.shape
    mask = torch.ones(S, S, dtype=torch.bool, device="cuda").triu(1)
    for b in range(B):
        for h in range(0, H, 1 if H < 40 else 5) if H % 5 else range(H):
            kv = h * k.shape[1] // H
            s = (q[b, h].double() @ k[b, kv].double().t() * D ** -0.5).masked_fill_(mask, float("-inf"))
            want = s.softmax(1) @ v[b, kv].double()
            rows = (o[b, h] - want).norm(dim=1) / want.norm(dim=1)
            assert (o[b, h] - want).norm() <= 5e-4 * want.norm() and rows.max() <= 2e-3, (b, h, rows.max(), rows.argmax())
            if lse is not None:
                assert ((lse[b, h] - s.logsumexp(1)).abs() <= 1e-3).all()


# four heads, two, one (with a third the group does not come out), and 18 workgroups for 71 heads
@pytest.mark.parametrize("B,Hq,Hkv,S,D", [(3, 32, 8, 769, 128), (4, 32, 8, 513, 128), (8, 36, 18, 257, 128), (6, 30, 10, 385, 128), (5, 16, 1, 895, 128),
                                          (3, 71, 1, 161, 64), (2, 71, 1, 299, 64), (2, 71, 71, 290, 64), (9, 34, 2, 159, 64), (1, 71, 1, 1025, 64)])
def test_heads_that_share_a_workgroup(B, Hq, Hkv, S, D):
    from triton_amd import ops
    g = torch.Generator().manual_seed(S)
    q, k, v = (ref.randn_half((B, h, S, D), g).cuda() for h in (Hq, Hkv, Hkv))
    o, lse = torch.full_like(q, 7.0), torch.zeros(B, Hq, S, device="cuda")
    assert ops.attention_kernel_name(q, k, v, o, D ** -0.5, True) == f"trn::attn_fwd16_kernel<{D}, 4, false>"
    ops.attention(q, k, v, o, D ** -0.5, True, lse=lse)
    compare(q, k, v, o, lse)


@pytest.mark.parametrize("D,B,Hq,Hkv,S", [(64, 2, 71, 1, 333), (128, 5, 32, 8, 460)])
def test_norms_and_given_queries(D, B, Hq, Hkv, S):
    from triton_amd import modules, ops
    g = torch.Generator().manual_seed(S)
    q, k, v = (ref.randn_half((B, h, S, D), g).cuda() for h in (Hq, Hkv, Hkv))
    o = torch.zeros_like(q)
    t = dict(Q=q, K=k, V=v, O=o, gamma_q=torch.ones(D, dtype=torch.half, device="cuda"), gamma_k=torch.ones(D, dtype=torch.half, device="cuda"))
    mod = modules.get("qknorm", eps=1e-5)
    mod.forward(*[t[p] for p in mod.TENSOR_PARAMS])
    norm = lambda x: (x.double() * (x.double().pow(2).mean(-1, keepdim=True) + 1e-5).rsqrt()).half()
    compare(norm(q), norm(k), v, o)
    n = torch.randn(B, Hq, S, S, device="cuda")
    need = ops.attention_key_scores_workspace_bytes(q, k, v, o, D ** -0.5, True, 3)
    ws = torch.empty(max(need, 256), dtype=torch.uint8, device="cuda")
    o.fill_(7.0)
    ops.attention_key_scores(q, k, v, o, D ** -0.5, True, torch.empty(B, Hq, S, device="cuda"), torch.empty(B, Hq, S, device="cuda"), noise=n, tau=1.0, workspace=ws)
    compare(q, k, v, o)


# short prompts whose last tile is nearly full: odd groups a head at a time, even ones in pairs, and the sizes on either side
@pytest.mark.parametrize("B,Hq,Hkv,S,D", [(6, 42, 2, 383, 64), (6, 42, 2, 352, 64), (4, 84, 2, 255, 128), (4, 35, 1, 256, 128), (6, 42, 2, 385, 64), (10, 35, 1, 353, 64)])
def test_groups_with_little_to_gain(B, Hq, Hkv, S, D):
    test_heads_that_share_a_workgroup(B, Hq, Hkv, S, D)
