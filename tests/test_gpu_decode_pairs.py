"""GPU parity of up to 32 queries whose keys are shared out in two launches, on both sides of the lines from which they are: shares
that see no key of a query, rows past the last query, workspaces with any contents.

Tolerance against float64: a probability and an output are rounded to fp16 once each, by 2^-11 / sqrt(3) of their size in root mean square at
most, 4.0e-4 in 2-norm; a row has up to twice that.  Row normalisers
are sums of the rounded probabilities, of 2000 and more of scores of standard deviation 1: 2^-11 / sqrt(3) x sqrt(e / 2000) = 1.04e-5 in root mean
square, asked for as six times that."""
import pytest
import torch

from oracle import ref

pytestmark = pytest.mark.gpu

# B, Hq, Hkv, Sq, Skv, D, causal, shared out
CASES = [
    (1, 8, 2, 16, 2000, 128, False, True), (1, 8, 2, 16, 1999, 128, False, False), (1, 32, 8, 32, 2245, 128, True, True),      # (2245: a last share of five keys)
    (1, 32, 32, 16, 2400, 128, True, True), (1, 32, 32, 16, 2399, 128, True, False), (1, 64, 8, 1, 3000, 128, True, True),
    (1, 120, 8, 5, 2716, 128, True, True), (1, 120, 8, 5, 2715, 128, True, False), (1, 128, 8, 5, 4000, 128, False, False),
    (1, 16, 16, 17, 2340, 64, True, True), (1, 16, 16, 17, 2339, 64, True, False), (1, 71, 1, 32, 2674, 64, True, True), (1, 71, 1, 32, 2673, 64, True, False),
    (1, 71, 71, 2, 7854, 64, True, True), (1, 71, 71, 2, 7853, 64, True, False), (3, 32, 4, 3, 3588, 64, True, True), (3, 32, 4, 3, 3587, 64, True, False),
    (2, 2, 1, 32, 3999, 128, True, True), (1, 8, 2, 33, 2500, 128, True, False),
    (1, 8, 2, 16, 4100, 128, True, None), (1, 4, 4, 32, 9997, 128, True, None), (1, 16, 4, 1, 12000, 64, True, None), (1, 71, 1, 9, 8193, 64, False, None),      # (their own workspace)
]


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,D,causal,shared", CASES)
def test_keys_shared_out_in_two_launches(B, Hq, Hkv, Sq, Skv, D, causal, shared):
    from triton_amd import ops
    g = torch.Generator().manual_seed(Skv)
    q, k, v = (ref.randn_half((B, h, s, D), g).cuda() for h, s in ((Hq, Sq), (Hkv, Skv), (Hkv, Skv)))
    scale = D ** -0.5
    o, plain = torch.full((B, Hq, 40, D), 7.0, dtype=torch.half, device="cuda"), torch.empty_like(q)
    need = ops.attention_chunk_workspace_bytes(q, k, v, plain, scale, causal)
    if shared is None:
        assert need == 0
        need = ops.attention_workspace_bytes(q, k, v, plain, scale, causal)
    assert (need > 0) == (shared is not False)
    ws = torch.full((max(need, 1024) + 512,), 255, dtype=torch.uint8, device="cuda")       # (NaN)
    lse, lse1 = torch.zeros(B, Hq, Sq, device="cuda"), torch.zeros(B, Hq, Sq, device="cuda")
    ops.attention(q, k, v, o[:, :, :Sq], scale, causal, lse=lse, workspace=ws)
    ops.attention(q, k, v, plain, scale, causal, lse=lse1)
    front = 512 if shared else (B * Hq + 63) // 64 * 256      # (counters of these heads; of any number in a workspace for chunks)
    assert (ws[:front] == 255).all() and (ws[max(need, 1024):] == 255).all() and (o[:, :, Sq:] == 7).all()
    assert (ws[512:need] != 255).any() == (shared is not False)
    small = torch.full((max(need - 256, 256),), 255, dtype=torch.uint8, device="cuda")
    again = torch.empty_like(q)
    ops.attention(q, k, v, again, scale, causal, workspace=small)
    assert torch.equal(again, plain) and (small == 255).all()
    mask = torch.ones(Sq, Skv, dtype=torch.bool, device="cuda").triu(Skv - Sq + 1)
    for b, h in {(0, 0), (B - 1, Hq - 1), (B // 2, Hq // 2)}:
        s = q[b, h].double() @ k[b, h * Hkv // Hq].double().t() * scale
        if causal:
            s = s.masked_fill(mask, float("-inf"))
        want = s.softmax(1) @ v[b, h * Hkv // Hq].double()
        rows = (o[b, h, :Sq] - want).norm(dim=1) / want.norm(dim=1)
        assert (o[b, h, :Sq] - want).norm() <= 4e-4 * want.norm() and rows.max() <= 8e-4, (rows.max(), rows.argmax())
        assert ((lse[b, h] - s.logsumexp(1)).abs() <= 6.2e-5).all() and ((lse1[b, h] - s.logsumexp(1)).abs() <= 6.2e-5).all()


# head_dim 64, as many KV heads, three shares: around the line of the launches without a workspace of their own (2600 + 74 x heads) and the
# 8192 keys from which that workspace is there: B, H, Sq, Skv
@pytest.mark.parametrize("B,H,Sq,Skv", [(1, 80, 2, 8192), (1, 80, 2, 8519), (1, 80, 2, 8520), (1, 76, 32, 8192), (1, 76, 1, 8224), (1, 85, 1, 8192), (1, 85, 1, 8889),
                                        (1, 85, 1, 8890), (5, 16, 16, 8519), (5, 16, 3, 8191)])
@pytest.mark.parametrize("causal", [False, True])
def test_what_the_workspace_held_before_does_not_matter(B, H, Sq, Skv, causal):
    """The workspace as allocated (zeros), full of NaN, with another call's shares in it, and the library's own after another call."""
    import ctypes as C
    from triton_amd import _lib, ops
    g = torch.Generator().manual_seed(Skv + H)
    D, scale = 64, 0.125
    q, k, v = (ref.randn_half((B, H, s, D), g).cuda() for s in (Sq, Skv, Skv))
    o = torch.zeros_like(q)
    need = ops.attention_workspace_bytes(q, k, v, o, scale, causal)
    assert (need > 0) == (Skv >= 8192)
    ws = torch.zeros(max(need, ops.attention_chunk_workspace_bytes(q, k, v, o, scale, causal), 256), dtype=torch.uint8, device="cuda")
    lib = _lib.load()

    def call(how, q, k, v, o, lse):
        if how != "own":
            return ops.attention(q, k, v, o, scale, causal, lse=lse, workspace=ws)
        d = ops._attn_desc(q, k, v, o, scale, causal, False, 0.0, None, 1.0)
        st = lib.trn_attn_fwd_noalloc_f16(C.byref(d), q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr(), None, None, None,
                                          torch.cuda.current_stream().cuda_stream)
        assert st == 0

    heads = [(0, 0), (B - 1, H - 1), (B // 2, H // 2)]
    mask = torch.ones(Sq, Skv, dtype=torch.bool, device="cuda").triu(Skv - Sq + 1)
    want = {}
    for b, h in heads:
        s = q[b, h].double() @ k[b, h].double().t() * scale
        if causal:
            s = s.masked_fill(mask, float("-inf"))
        want[b, h] = s.softmax(1) @ v[b, h].double(), s.logsumexp(1)
    first = None
    for how in ("zeros", "nan", "used", "own"):
        if how == "nan":
            ws.fill_(255)
        elif how in ("used", "own"):                    # another problem's results in the same places: keys twice as large, other values
            call(how, q, k * 2, v + 8, torch.zeros_like(q), torch.zeros(B, H, Sq, device="cuda"))
        o, lse = torch.full_like(q, 7.0), torch.full((B, H, Sq), 7.0, device="cuda")
        call(how, q, k, v, o, lse)
        for at in heads:
            w, l = want[at]
            assert (o[at] - w).norm() <= 4e-4 * w.norm() and ((lse[at] - l).abs() <= 6.2e-5).all(), how
        if need > 0:                                    # (the library's own serves the same shares)
            first = first or (o, lse)
            assert torch.equal(o, first[0]) and torch.equal(lse, first[1]), how


@pytest.mark.parametrize("D", [64, 128])
def test_one_workspace_for_counters_and_chunks(D):
    """One zero-filled workspace: keys shared out in two launches, then a call with noise of more heads, whose counters have to be zero still."""
    from triton_amd import ops
    g = torch.Generator().manual_seed(D)
    scale = D ** -0.5
    q, k, v = (ref.randn_half((1, 71, s, D), g).cuda() for s in (2, 8200, 8200))
    noise = torch.randn(1, 71, 2, 8200, generator=g).cuda()
    few = [t[:, :32, :2, :].contiguous() if t is q else t[:, :32, :3700].contiguous() for t in (q, k, v)]
    o, o1 = torch.full_like(q, 7.0), torch.full_like(q, 7.0)
    lse, lse1 = torch.full((1, 71, 2), 7.0, device="cuda"), torch.full((1, 71, 2), 7.0, device="cuda")
    small = ops.attention_chunk_workspace_bytes(*few, torch.zeros_like(few[0]), scale, True)
    big = ops.attention_workspace_bytes(q, k, v, o, scale, True)
    assert small > 0 and big > 0
    ws = torch.zeros(max(small, big), dtype=torch.uint8, device="cuda")
    ops.attention(q, k, v, o, scale, True, noise=noise, tau=1.0, lse_pert=lse, workspace=ws)
    got, alone = torch.zeros_like(few[0]), torch.zeros_like(few[0])
    ops.attention(*few, got, scale, True, workspace=ws)
    ops.attention(*few, alone, scale, True)
    assert not torch.equal(got, alone) and (got.double() - alone.double()).norm() <= 8e-4 * alone.double().norm()      # (shared out)
    assert (ws[:512] == 0).all()
    for _ in range(2):
        ops.attention(q, k, v, o1, scale, True, noise=noise, tau=1.0, lse_pert=lse1, workspace=ws)
        assert torch.equal(o, o1) and torch.equal(lse, lse1)
        o1.fill_(7.0)


# 2245 and 4100 keys: shares of 288 (the last of 5) and of 320 (of 260); 8200 of 64 with its own workspace, shares of 1056
@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,D", [(1, 32, 8, 17, 2245, 128), (1, 8, 2, 32, 4100, 128), (1, 16, 16, 1, 2400, 64), (1, 71, 1, 5, 8200, 64)])
@pytest.mark.parametrize("first,last", [(0, None), (0, 400), (1056, 2200), (-3, None), (-300, None)])
def test_scores_that_are_no_numbers(B, Hq, Hkv, Sq, Skv, D, first, last):
    """NaN keys in a part of a share, in a whole one and in several, and a NaN query: the same outputs and normalisers are NaN as without shares."""
    from triton_amd import ops
    g = torch.Generator().manual_seed(Skv)
    q, k, v = (ref.randn_half((B, h, s, D), g).cuda() for h, s in ((Hq, Sq), (Hkv, Skv), (Hkv, Skv)))
    k[:, 0, first:last] = float("nan")
    q[:, -1, Sq // 2] = float("nan")
    scale, outs = D ** -0.5, []
    need = max(ops.attention_workspace_bytes(q, k, v, q, scale, True), ops.attention_chunk_workspace_bytes(q, k, v, q, scale, True))
    assert need > 0
    for ws in (None, torch.zeros(need, dtype=torch.uint8, device="cuda")):
        o, lse = torch.full_like(q, 7.0), torch.full((B, Hq, Sq), 7.0, device="cuda")
        ops.attention(q, k, v, o, scale, True, lse=lse, workspace=ws)
        outs.append((o, lse))
    (o1, l1), (o2, l2) = outs
    visible = torch.arange(Skv, device="cuda")[None] <= torch.arange(Sq, device="cuda")[:, None] + Skv - Sq
    poisoned = torch.zeros(Skv, dtype=torch.bool, device="cuda")
    poisoned[first:last] = True
    rows = torch.zeros(B, Hq, Sq, dtype=torch.bool, device="cuda")
    rows[:, :Hq // Hkv] = (visible & poisoned).any(1)
    rows[:, -1, Sq // 2] = True
    assert torch.equal(o1.isnan().all(3), rows) and torch.equal(l1.isnan(), rows)
    assert torch.equal(o1.isnan(), o2.isnan()) and torch.equal(l1.isnan(), l2.isnan())
    d = (o1 - o2)[~rows].double()
    assert d.norm() <= 8e-4 * o1[~rows].double().norm() and ((l1 - l2)[~rows].abs() <= 1.24e-4).all()      # (twice the distance of each from float64)


# KV groups that the 8 XCDs do not share evenly -- two shares where there is room for three, four of six, none yet --, and long caches: B, Hq, Hkv, Sq,
# Skv, D, causal, shared out, as above
@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,D,causal,shared", [
    (1, 72, 9, 4, 3600, 64, True, True), (1, 72, 9, 4, 3599, 64, True, False), (2, 21, 3, 9, 3041, 128, False, True), (1, 42, 21, 9, 3040, 128, True, True),
    (1, 42, 21, 9, 3039, 128, True, False), (1, 100, 25, 2, 6000, 64, True, True), (1, 100, 25, 2, 5999, 64, True, False), (1, 122, 61, 3, 8191, 128, True, False),
    (1, 122, 61, 3, 8192, 128, True, None), (1, 38, 38, 32, 16000, 64, True, None), (1, 70, 10, 1, 10001, 64, False, None), (1, 36, 6, 17, 9000, 128, True, None),
])
def test_keys_of_uneven_groups(B, Hq, Hkv, Sq, Skv, D, causal, shared):
    test_keys_shared_out_in_two_launches(B, Hq, Hkv, Sq, Skv, D, causal, shared)
