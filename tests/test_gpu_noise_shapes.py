"""GPU parity of the KeyFormer pair (forward with score perturbation, key statistics) in the workgroup shapes and cache policies
of the forward, with the noise at every row alignment: keys split over two groups of waves, 128 and 256 queries a workgroup.

Tolerances: outputs to 2e-3 of each query's 2-norm (fp16 probabilities and one fp16 rounding, 2^-11 each at most, are some 3e-4 of a
norm; an element of an output is 0.02 to 0.05 at these lengths, so that an absolute bound of that size would see nothing),
1e-3 relative on fp32 key scores as in test_gpu_scores.py."""
import pytest
import torch

from oracle import ref

pytestmark = pytest.mark.gpu

FWD = "attn_fwd_kernel<{}, {}, true>"           # in the cache policy of the shape's usual sizes
OTHER = "attn_fwd_kernel<{}, {}, false>"
SPLIT = "attn_fwd_split_kernel<{}, false, false>"

# B, Hq, Hkv, S, D, fp16 noise, spare elements per noise row, first element, kernel by the launch rule
CASES = [
    (1, 27, 9, 577, 128, False, 3, 0, SPLIT.format(128)), (1, 27, 9, 577, 128, True, 0, 1, SPLIT.format(128)),     # odd rows, a tile of 65
    (1, 26, 2, 640, 128, True, 0, 0, SPLIT.format(128)), (2, 14, 7, 641, 128, False, 0, 1, SPLIT.format(128)),     # whole tiles, and one row more
    (1, 16, 4, 1025, 64, True, 0, 0, SPLIT.format(64)), (1, 16, 16, 1152, 64, False, 0, 0, SPLIT.format(64)),
    (1, 64, 8, 600, 128, True, 1, 0, FWD.format(128, 4)), (1, 71, 1, 250, 64, True, 0, 1, FWD.format(64, 4)),      # shared CUs
    (1, 71, 1, 257, 64, False, 2, 1, FWD.format(64, 4)), (4, 32, 8, 512, 128, False, 0, 0, FWD.format(128, 4)),
    (2, 33, 11, 1282, 128, True, 1, 1, FWD.format(128, 8)), (2, 33, 11, 1290, 128, False, 0, 3, OTHER.format(128, 8)),
]


def noise_tensor(B, H, S, half, spare, first, seed):
    """Gumbel noise [B, H, S, S] inside rows of S + spare elements that begin `first` elements into the storage; NaN elsewhere."""
    pitch = S + spare
    flat = torch.full((B * H * S * pitch + first,), float("nan"), dtype=torch.float16 if half else torch.float32, device="cuda")
    n = torch.as_strided(flat, (B, H, S, S), (H * S * pitch, S * pitch, pitch, 1), first)
    g = torch.Generator(device="cuda").manual_seed(seed)
    for b in range(B):
        for h in range(H):
            n[b, h] = -torch.log(torch.empty(S, S, device="cuda").exponential_(generator=g))
    return n


def run(q, k, v, noise, scale, tau):
    """The two launches by themselves: without a workspace the single pass over the noise is not taken (but where a head has one
    workgroup, which takes some 240 heads)."""
    from triton_amd import ops
    assert q.shape[0] * q.shape[1] <= 128
    c = torch.full(q.shape[:3], -1.0, dtype=torch.float32, device="cuda")
    o = torch.full_like(q, 7.0)
    ops.attention_key_scores(q, k, v, o, scale, True, torch.empty_like(c), c, noise=noise, tau=tau)
    torch.cuda.synchronize()
    return o, c


def through_the_module(q, k, v, noise, tau):
    from triton_amd import modules
    c, o = torch.full(q.shape[:3], -1.0, dtype=torch.float32, device="cuda"), torch.full_like(q, 7.0)
    m = modules.get("keyformer", tau=tau)
    t = dict(Q=q, K=k, V=v, O=o, noise=noise, C_out=c)
    m.forward(*[t[p] for p in m.TENSOR_PARAMS])
    torch.cuda.synchronize()
    return o, c


@pytest.mark.parametrize("B,Hq,Hkv,S,D,half,spare,first,name", CASES)
def test_keyformer_in_every_shape_and_row_alignment(B, Hq, Hkv, S, D, half, spare, first, name):
    from triton_amd import ops
    g = torch.Generator().manual_seed(S + D)
    q, k, v = (ref.randn_half((B, h, S, D), g).cuda() for h in (Hq, Hkv, Hkv))
    noise = noise_tensor(B, Hq, S, half, spare, first, S)
    scale, tau = D ** -0.5, 1.5
    # (the function speaks for fp32 noise: of the kernel for fp16 it gives the shape)
    launched = ops.attention_kernel_name(q, k, v, torch.empty_like(q), scale, True, half or noise)
    assert launched.rsplit(",", 1)[0] == "trn::" + name.rsplit(",", 1)[0] and (half or launched == "trn::" + name)
    o, c = run(q, k, v, noise, scale, tau)
    if ops.attention_key_scores_workspace_bytes(q, k, v, o, scale, True, 2 if half else 3) == 0:       # (elsewhere the module takes the single pass)
        assert all(torch.equal(x, y) for x, y in zip((o, c), through_the_module(q, k, v, noise, tau)))
    keep = torch.ones(S, S, dtype=torch.bool, device="cuda").tril()
    for b in range(B):
        for h in range(Hq):
            s = (q[b, h].float() @ k[b, h * Hkv // Hq].float().T * scale).masked_fill(~keep, float("-inf"))
            want = s.softmax(-1) @ v[b, h * Hkv // Hq].float()
            err = ((o[b, h].float() - want).norm(dim=-1) / want.norm(dim=-1)).max()
            assert err <= 2e-3, f"batch {b} head {h}: a query's output off by {err:.3g} of its norm"
            want = ((s + noise[b, h].float().masked_fill(~keep, 0)) / tau).softmax(-1).sum(0)
            rel = ((c[b, h] - want).abs() / want).max()
            assert rel < 1e-3, f"batch {b} head {h}: scores off by {rel:.3g} relative"


@pytest.mark.parametrize("H,Hkv,S,D", [(32, 8, 1792, 128), (32, 8, 2048, 128), (32, 8, 3072, 128), (71, 1, 1536, 64), (16, 16, 2560, 64)])
def test_noise_past_the_caches_gives_the_same_bits(H, Hkv, S, D):
    """Rows on whole 128-byte lines and too much noise for the last-level cache: requested with the non-temporal hint.  The same
    values four elements further on are not."""
    g = torch.Generator(device="cuda").manual_seed(S)
    q, k, v = (torch.randn(1, h, S, D, generator=g, device="cuda").half() for h in (H, Hkv, Hkv))
    store = torch.empty(H * S * S + 32, device="cuda")
    base = (-store.data_ptr() // 4) % 32
    results = []
    for first in (base, (base + 4) % 32):
        noise = torch.as_strided(store, (1, H, S, S), (H * S * S, S * S, S, 1), first)
        gn = torch.Generator(device="cuda").manual_seed(5)
        for h in range(H):
            noise[0, h] = -torch.log(torch.empty(S, S, device="cuda").exponential_(generator=gn))
        results.append(run(q, k, v, noise, D ** -0.5, 1.0))
    for a, b in zip(*results):
        assert torch.equal(a, b)
