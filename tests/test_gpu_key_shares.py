"""A chunk of queries on a long cache with the keys shared out over workgroups (trn_attn_chunk_workspace_bytes), against the
float64 softmax: query tiles and key shares with remainders, the causal diagonal inside a share and shares that some or all
queries of a tile do not see, GQA, the fused query norm, the row normalisers."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def chunk_bytes(q, k, o, scale, causal):
    import ctypes as C
    from triton_amd import _lib, ops
    d = ops._attn_desc(q, k, k, o, scale, causal, False, 0.0, None, 1.0)
    return int(_lib.load().trn_attn_chunk_workspace_bytes(C.byref(d)))


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,D,causal,q_norm", [
    (1, 8, 2, 33, 3072, 128, True, False), (1, 8, 8, 128, 3073, 128, False, True), (2, 3, 1, 129, 3199, 128, True, False),
    (1, 4, 2, 700, 4159, 64, True, False), (1, 71, 1, 100, 2600, 64, True, True), (1, 32, 32, 257, 3200, 128, True, False),
    (1, 1, 1, 2300, 4200, 64, True, False), (1, 2, 1, 3100, 3100, 128, True, False), (1, 64, 8, 40, 4097, 64, False, False)])
def test_shared_out_keys(B, Hq, Hkv, Sq, Skv, D, causal, q_norm):
    """Element by element 4e-3 + 1e-3 of the value, as the other attention kernels are held to on N(0,1) inputs (one fp16 rounding
    each of the normalised Q, of the probabilities and of the result), so that late rows, whose results are averages over
    thousands of keys and small, count like the first ones; row normalisers 2e-3."""
    from triton_amd import ops
    g = torch.Generator(device="cuda").manual_seed(3)
    q, k, v = (torch.randn(B, h, s, D, generator=g, device="cuda").half() for h, s in ((Hq, Sq), (Hkv, Skv), (Hkv, Skv)))
    o, lse, scale = torch.zeros_like(q), torch.zeros(B, Hq, Sq, device="cuda"), D ** -0.5
    n = chunk_bytes(q, k, o, scale, causal)
    assert n > 0
    ws = torch.full((n + 64,), 0xFF, dtype=torch.uint8, device="cuda")             # (NaN wherever it is not written first)
    ops.attention(q, k, v, o, scale, causal, lse=lse, q_norm=q_norm, q_eps=1e-5, workspace=ws[:n])
    again, short, plain = torch.zeros_like(q), torch.zeros_like(q), torch.zeros_like(q)
    ops.attention(q, k, v, again, scale, causal, q_norm=q_norm, q_eps=1e-5, workspace=ws[:n])
    ops.attention(q, k, v, short, scale, causal, q_norm=q_norm, q_eps=1e-5, workspace=ws[:n - 256])   # too small: not used
    ops.attention(q, k, v, plain, scale, causal, q_norm=q_norm, q_eps=1e-5)
    torch.cuda.synchronize()
    assert torch.equal(o, again) and torch.equal(short, plain)
    assert bool((ws[n:] == 0xFF).all())
    for b in range(B):
        for h in range(Hq):
            x = q[b, h].double()
            if q_norm:
                x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-5)
            s = x @ k[b, h // (Hq // Hkv)].double().T * scale
            if causal:
                s = s.masked_fill(~torch.ones(Sq, Skv, dtype=torch.bool, device="cuda").tril(Skv - Sq), float("-inf"))
            want = s.softmax(-1) @ v[b, h // (Hq // Hkv)].double()
            for got in (o, plain):
                assert ((got[b, h].double() - want).abs() <= 4e-3 + 1e-3 * want.abs()).all(), (b, h)
            assert (lse[b, h].double() - torch.logsumexp(s, -1)).abs().max() < 2e-3, (b, h)


def test_which_problems_share_out_their_keys():
    """One side and the other of each bound of the rule; the size does not depend on the number of keys."""
    def need(heads, sq, skv, D):
        q, k = torch.empty(1, heads, sq, D, dtype=torch.float16, device="cuda"), torch.empty(1, 1, skv, D, dtype=torch.float16, device="cuda")
        return chunk_bytes(q, k, q, 1.0, True)
    assert need(8, 32, 8192, 128) == 0 and need(8, 33, 8192, 128) == need(8, 33, 3072, 128) == 512 + 8 * 16 * 33 * 130 * 4
    assert need(8, 33, 3071, 128) == 0 and need(8, 33, 4095, 64) == 0 and need(8, 33, 4096, 64) == 512 + 8 * 16 * 33 * 66 * 4
    assert need(71, 100, 2560, 64) == 512 + 71 * 3 * 100 * 66 * 4 and need(71, 100, 2559, 64) == 0 and need(71, 64, 2560, 64) == 0
    assert need(128, 128, 4096, 128) > 0 and need(129, 128, 4096, 128) == 0


def test_one_workspace_for_chunks_and_single_tokens():
    """The split decode shapes find their arrival counters as they left them, whatever a chunk wrote in between."""
    from triton_amd import ops
    g = torch.Generator(device="cuda").manual_seed(5)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").half()
    k, v, chunk, one = r(1, 8, 5000, 128), r(1, 8, 5000, 128), r(1, 8, 100, 128), r(1, 8, 1, 128)
    n = max(chunk_bytes(chunk, k, chunk, 0.1, False), ops.attention_workspace_bytes(one, k, v, one, 0.1, False))
    ws, want, got = torch.zeros(n, dtype=torch.uint8, device="cuda"), torch.zeros_like(one), torch.zeros_like(one)
    ops.attention(one, k, v, want, 0.1, False, workspace=torch.zeros_like(ws))
    ops.attention(chunk, k, v, torch.zeros_like(chunk), 0.1, False, workspace=ws)
    assert not ws[:512].any()
    ops.attention(one, k, v, got, 0.1, False, workspace=ws)
    torch.cuda.synchronize()
    assert torch.equal(got, want)
