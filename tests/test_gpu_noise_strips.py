"""GPU parity of KeyFormer's prompts whose row normalisers and key scores come from one pass over the noise (32 queries at a
time, their exponentials kept in registers): held keys and those beyond, strips and blocks cut off by the end, noise at every
row alignment, references that have to rise.

Tolerance on the scores against float64: their exponents z are good to a few roundings of |z| log2 e in fp32 (2^-24 relative
each), a probability to 4 x 2^-24 x |z| ln 2, some 5e-6 at |z| = 30 and 1.7e-4 at 1000; the sums over queries add less than that.  The row normalisers: as the
exponents, 3e-7 of the largest |z| (a reference that rises by as much leaves its rounding), and a rounding of what lies around 1."""
import pytest
import torch

from oracle import ref

pytestmark = pytest.mark.gpu


def problem(B, Hq, Hkv, S, D, half, spare, first, seed=1):
    g = torch.Generator().manual_seed(seed + S)
    q, k, v = (ref.randn_half((B, h, S, D), g).cuda() for h in (Hq, Hkv, Hkv))
    pitch = S + spare
    flat = torch.full((B * Hq * S * pitch + first,), float("nan"), dtype=torch.float16 if half else torch.float32, device="cuda")
    n = torch.as_strided(flat, (B, Hq, S, S), (Hq * S * pitch, S * pitch, pitch, 1), first)
    gg = torch.Generator(device="cuda").manual_seed(seed)
    for b in range(B):
        n[b] = -torch.log(torch.empty(Hq, S, S, device="cuda").exponential_(generator=gg))
    return q, k, v, n


def scores(q, k, v, n, tau, with_workspace=True, one_workgroup=False, out=torch.float32):
    from triton_amd import ops
    B, H, S, D = q.shape
    o, rows, c = torch.empty_like(q), torch.full((B, H, S), 9.0, device="cuda"), torch.full((B, H, S), -1.0, dtype=out, device="cuda")
    need = ops.attention_key_scores_workspace_bytes(q, k, v, o, D ** -0.5, True, 2 if n.dtype == torch.half else 3)
    assert (need == 0) == one_workgroup          # (one workgroup a head needs none)
    ws = torch.full((need,), 255, dtype=torch.uint8, device="cuda") if with_workspace else None      # (any contents: NaN here)
    ops.attention_key_scores(q, k, v, o, D ** -0.5, True, rows, c, noise=n, tau=tau, workspace=ws)
    torch.cuda.synchronize()
    return o, rows, c


def check(q, k, n, rows, c, tau, tol, heads, largest=0.0):
    B, H, S, D = q.shape
    mask = torch.ones(S, S, dtype=torch.bool, device="cuda").triu(1)
    for b, h in heads:
        z = (q[b, h].double() @ k[b, h * k.shape[1] // H].double().t() * D ** -0.5 + n[b, h].double()) / tau
        z.masked_fill_(mask, float("-inf"))
        lse = z.logsumexp(1)
        want = (z - lse[:, None]).exp().sum(0)
        assert ((rows[b, h] - lse).abs() <= 4e-6 + 3e-7 * lse.abs().clamp(min=largest)).all(), (rows[b, h] - lse).abs().max()
        assert ((c[b, h] - want).abs() <= tol * want + 1e-30).all(), ((c[b, h] - want).abs() / want).max()


def check_outputs(q, k, v, o, heads):
    """O of these heads against float64: the probabilities and the outputs are rounded to fp16 once each, by 2^-11 / sqrt(3) of their
    size in root mean square at most and independently of each other: sqrt(2) times that, 4.0e-4, in 2-norm (measured 2.1e-4 to
    2.6e-4).  Queries rounded once more after the scale go past it: 6.1e-4 for scores of standard deviation 8."""
    S, D = q.shape[2:]
    mask = torch.ones(S, S, dtype=torch.bool, device="cuda").triu(1)
    for b, h in heads:
        kv = h * k.shape[1] // q.shape[1]
        p = (q[b, h].double() @ k[b, kv].double().t() * D ** -0.5).masked_fill_(mask, float("-inf")).softmax(1)
        want = p @ v[b, kv].double()
        assert (o[b, h] - want).norm() <= 4e-4 * want.norm(), (o[b, h] - want).norm() / want.norm()


# B, Hq, Hkv, S, D, kernel of the attention without noise
SHAPES = [
    (1, 32, 8, 401, 128, "attn_fwd16_kernel<128, 4, false>"), (1, 71, 1, 609, 64, "attn_fwd16_kernel<64, 4, false>"),
    (1, 8, 2, 2050, 128, "attn_fwd16_split_kernel<128>"), (1, 16, 16, 1101, 64, "attn_fwd16_split_kernel<64>"),
    (1, 32, 8, 1500, 128, "attn_fwd16_kernel<128, 8, true>"), (1, 32, 8, 1535, 64, "attn_fwd16_kernel<64, 8, true>"),
    (2, 24, 6, 2040, 128, "attn_fwd16_kernel<128, 8, false>"),
]


@pytest.mark.parametrize("large", [1, 8])
@pytest.mark.parametrize("B,Hq,Hkv,S,D,kernel", SHAPES)
def test_outputs_from_queries_as_given(B, Hq, Hkv, S, D, kernel, large):
    """The attention beside the single pass keeps the queries as they are given, in each workgroup shape, as the forward with noise
    does, also where scores are large."""
    from triton_amd import ops
    q, k, v, n = problem(B, Hq, Hkv, S, D, False, 0, 0, seed=7)
    q *= large
    assert ops.attention_kernel_name(q, k, v, q, D ** -0.5, True) == "trn::" + kernel
    o, _, _ = scores(q, k, v, n, 1.0)
    check_outputs(q, k, v, o, [(0, 0), (B - 1, Hq - 1), (B // 2, Hq // 3)])


# B, Hq, Hkv, S, D, fp16 noise, spare elements per row, first element
CASES = [
    (2, 72, 1, 321, 64, False, 0, 0), (4, 64, 8, 353, 64, False, 3, 1), (1, 71, 1, 352, 64, True, 0, 0), (1, 71, 71, 351, 64, True, 1, 1),
    (3, 32, 8, 351, 128, False, 1, 0), (1, 32, 8, 321, 128, True, 0, 1), (1, 32, 8, 300, 128, True, 3, 1), (1, 32, 4, 415, 128, False, 0, 0),    # strips and blocks cut short
    (1, 8, 2, 800, 128, True, 0, 0), (2, 32, 8, 625, 128, True, 1, 1), (1, 16, 16, 703, 64, True, 0, 0), (1, 16, 4, 737, 64, False, 0, 0),    # the rule's lines
    (2, 24, 6, 1024, 128, False, 0, 0), (1, 32, 8, 1057, 128, True, 0, 1), (1, 40, 8, 1056, 64, False, 32, 0),     # at the end of the held keys
    (1, 4, 1, 2048, 64, False, 0, 0), (1, 5, 5, 2081, 64, False, 0, 2), (1, 8, 2, 2305, 128, True, 1, 0), (1, 6, 3, 2113, 128, False, 3, 0),
    (1, 3, 1, 4193, 128, False, 0, 0), (1, 2, 2, 4830, 64, True, 2, 1),                        # the longest rows
]


@pytest.mark.parametrize("B,Hq,Hkv,S,D,half,spare,first", CASES)
def test_one_pass_over_the_noise(B, Hq, Hkv, S, D, half, spare, first):
    tau = 1.5
    q, k, v, n = problem(B, Hq, Hkv, S, D, half, spare, first)
    o, rows, c = scores(q, k, v, n, tau)
    heads = [(0, 0), (B - 1, Hq - 1), (B // 2, Hq // 2)]
    check(q, k, n, rows, c, tau, 2e-5, heads)
    check_outputs(q, k, v, o, heads)
    # a second call gives the same bits
    o2, rows2, c2 = scores(q, k, v, n, tau)
    assert torch.equal(rows, rows2) and torch.equal(c, c2) and torch.equal(o, o2)
    # without the workspace: forward and statistics with a pass each
    o1, rows1, c1 = scores(q, k, v, n, tau, with_workspace=False)
    assert ((o1 - o).float().norm(dim=-1) <= 4e-3 * o.float().norm(dim=-1)).all()
    assert (c1 - c).norm() <= 1e-4 * c.norm() and (rows1 - rows).abs().max() < 1e-3


@pytest.mark.parametrize("B,Hq,Hkv,S,D,half,one", [(6, 71, 1, 333, 64, False, True), (6, 71, 1, 633, 64, True, True), (8, 64, 8, 401, 128, False, True), (4, 64, 8, 1650, 64, True, True),
                                                   (1, 71, 1, 333, 64, False, False), (1, 32, 8, 701, 128, True, False)])
def test_one_workgroup_a_head_and_scores_in_half(B, Hq, Hkv, S, D, half, one):
    """A head of one workgroup, which writes its column sums itself, and several, whose sums a second launch adds; as fp16 the
    fp32 scores rounded once in both.  The row normalisers do not depend on how many there are: those of one batch entry alone, whose heads have several
    workgroups, are the same bits (those of the two passes are not)."""
    q, k, v, n = problem(B, Hq, Hkv, S, D, half, 1, 1, seed=9)
    o, rows, c = scores(q, k, v, n, 1.5, with_workspace=not one, one_workgroup=one)
    check(q, k, n, rows, c, 1.5, 2e-5, [(0, 0), (B - 1, Hq - 1), (B // 2, Hq // 2)])
    check_outputs(q, k, v, o, [(0, 0), (B - 1, Hq - 1)])
    _, rows16, c16 = scores(q, k, v, n, 1.5, with_workspace=not one, one_workgroup=one, out=torch.half)
    assert torch.equal(c16, c.half()) and torch.equal(rows16, rows)
    if one:
        _, rows1, c1 = scores(q[-1:], k[-1:], v[-1:], n[-1:], 1.5)
        assert torch.equal(rows1, rows[-1:]) and (c1 - c[-1:]).abs().max() <= 1e-5 * c.abs().max()


def test_workspaces_of_many_lengths():
    """Prompts of every length in an instance share the workspaces of the single pass: powers of two, so that all of them hold at
    most twice the largest of them, and none where a head has one workgroup."""
    from triton_amd import modules, ops
    m, most = modules.get("keyformer"), 0
    q = torch.randn(1, 8, 2400, 128, device="cuda").half()
    kv = torch.randn(1, 2, 2400, 128, device="cuda").half()
    n = torch.randn(8 * 2400 * 2400, device="cuda").half()
    for S in list(range(801, 2400, 97)):
        t = dict(Q=q[:, :, :S].contiguous(), K=kv[:, :, :S].contiguous(), V=kv[:, :, :S].contiguous(), O=torch.empty(1, 8, S, 128, dtype=torch.half, device="cuda"),
                 noise=n[: 8 * S * S].view(1, 8, S, S), C_out=torch.empty(1, 8, S, dtype=torch.half, device="cuda"))
        m.forward(*[t[p] for p in m.TENSOR_PARAMS])
        most = max(most, ops.attention_key_scores_workspace_bytes(t["Q"], t["K"], t["V"], t["O"], 0.1, True, 2))
    sizes = [w.numel() for key, w in m._ws.items() if key[0] == "key_parts"]
    assert most > 1 << 20 and sizes and all(x & (x - 1) == 0 for x in sizes) and sum(sizes) <= 4 * most
    m = modules.get("keyformer")
    t = dict(Q=torch.randn(6, 71, 333, 64, device="cuda").half(), K=torch.randn(6, 1, 333, 64, device="cuda").half(), V=torch.randn(6, 1, 333, 64, device="cuda").half(),
             O=torch.empty(6, 71, 333, 64, dtype=torch.half, device="cuda"), noise=torch.randn(6, 71, 333, 333, device="cuda"), C_out=torch.empty(6, 71, 333, device="cuda"))
    m.forward(*[t[p] for p in m.TENSOR_PARAMS])
    torch.cuda.synchronize()
    assert not [key for key in m._ws if key[0] == "key_parts"]


@pytest.mark.parametrize("S,D,Hq", [(1100, 128, 32), (2200, 64, 8), (1090, 64, 71)])
def test_references_that_rise_and_rows_without_noise(S, D, Hq):
    """Scores that jump by hundreds within a row, before and beyond the held keys; keys that are all but masked (-1000), keys that
    are (-inf), from the first one on, for some rows of a strip and for all."""
    q, k, v, n = problem(1, Hq, Hq, S, D, False, 0, 0, seed=3)
    n[0, 0, :, 40:] += 300.0
    n[0, 0, :, S // 2:] += 300.0
    n[0, 1, :, :200] = -1e3
    n[0, 1, 3::5, :10] = 0.0
    n[0, 2, 300:, :299] = float("-inf")
    n[0, 2, 7::3, 20:260] = float("-inf")
    n[0, 3, :, ::2] += 500.0
    o, rows, c = scores(q, k, v, n, 1.0)
    check(q, k, n, rows, c, 1.0, 4e-4, [(0, h) for h in range(5)], 1000.0)


@pytest.mark.parametrize("S,D,Hq,half,mask", [(1100, 128, 32, False, -1e4), (1100, 64, 71, False, -1e9), (2200, 64, 8, False, -1e9), (2200, 64, 8, False, -1e30), (2200, 64, 8, True, -65504.0),
                                              (1030, 64, 71, True, -1e4), (3100, 64, 4, False, -1e6)])
def test_keys_masked_by_finite_numbers(S, D, Hq, half, mask):
    """Keys that later rows are kept from by a large negative number, whole blocks of them and the first that some waves see among
    these, before the held keys (2200, 3100) and within: the scores of the others are as exact as without.  (A reference of -1e9
    has a last place of 64.)"""
    q, k, v, n = problem(1, Hq, Hq, S, D, half, 0, 0, seed=11)
    for h, first in enumerate((0, 32, 100, 1)):
        n[0, h, 400:, first:400] = mask
    n[0, 3, 700:, 400:640] = mask
    n[0, 3, 900::3, 128:800] = mask
    o, rows, c = scores(q, k, v, n, 1.0)
    check(q, k, n, rows, c, 1.0, 2e-5, [(0, h) for h in range(4)])


@pytest.mark.parametrize("S,D,Hq,half", [(1100, 128, 32, False), (620, 64, 71, False), (2200, 64, 8, False), (1030, 64, 71, True)])
def test_rows_without_a_normaliser(S, D, Hq, half):
    """A row without a finite score, or with +inf or NaN among them, has no probabilities: the scores of the keys that it sees are
    NaN, and only these.  A row whose scores are all the same huge negative number is uniform as long as that is finite (and its keys
    held; beyond them the last place of the normaliser is more than log n).  At 6e4 the exponents of a row's first block, which has
    no reference yet, are rounded to 2^-8 and the probabilities to 2^-8 of themselves."""
    r = 300
    for what in ("-inf", "+inf", "nan", "low"):
        q, k, v, n = problem(1, Hq, Hq, S, D, half, 0, 0, seed=5)
        _, _, base = scores(q, k, v, n, 1.0)
        seen = lambda: (n[0, 0, r].double() + k[0, 0].double() @ q[0, 0, r].double() * D ** -0.5)[: r + 1].softmax(0)
        before = seen()
        if what == "low":
            n[0, 0, r] = -6e4 if half else -1e38
        elif what == "-inf":
            n[0, 0, r] = float("-inf")
        else:
            n[0, 0, r, 5] = float(what)
        _, rows, c = scores(q, k, v, n, 1.0)
        assert torch.equal(c[:, 1:], base[:, 1:])
        assert ((c[0, 0, r + 1:] - base[0, 0, r + 1:]).abs() <= 2e-5 * base[0, 0, r + 1:]).all(), what
        if what == "low":
            want = base[0, 0, : r + 1].double() - before + seen()
            assert ((c[0, 0, : r + 1] - want).abs() <= 2e-5 * want + (2.0 ** -7 * seen() if half else 0)).all()
        else:
            assert c[0, 0, : r + 1].isnan().all(), what


@pytest.mark.parametrize("general", [False, True])
def test_capture_with_noise_of_the_other_type(general):
    """One eager call per shape is what a capture needs, with noise of either type: where only fp16 noise has the single pass, a
    capture with it after an eager call with fp32 noise goes without its workspace, in two passes.  general: scores that the kernels
    do not write themselves (the path in Python)."""
    from triton_amd import modules
    q, k, v, n = problem(1, 8, 2, 1000, 128, True, 0, 0)
    c, o = torch.empty(1, 8, 2000, dtype=torch.half, device="cuda")[..., ::2] if general else torch.empty(1, 8, 1000, dtype=torch.half, device="cuda"), torch.empty_like(q)
    m = modules.get("keyformer")
    t = dict(Q=q, K=k, V=v, O=o, noise=n.float(), C_out=c)
    m.forward(*[t[p] for p in m.TENSOR_PARAMS])
    t["noise"] = n
    args = [t[p] for p in m.TENSOR_PARAMS]
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        m.forward(*args)
    for _ in range(3):
        c.fill_(-1.0); o.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        check_outputs(q, k, v, o, [(0, 0), (0, 7)])
        rows = torch.stack([((q[0, h].double() @ k[0, h // 4].double().t() * 128 ** -0.5 + n[0, h].double())
                             .masked_fill(torch.ones(1000, 1000, dtype=torch.bool, device="cuda").triu(1), float("-inf"))).softmax(1).sum(0) for h in range(8)])
        assert ((c[0] - rows).abs() <= 2.0 ** -11 * rows + 2e-5 * rows + 2.0 ** -24).all()


def test_captured_module_and_where_the_rule_lies():
    from triton_amd import modules, ops
    # from 300 keys and some MB of noise; the workspace serves either type
    def need(B, H, S, D, causal=True, Skv=None, noise=True):
        q, k = (torch.as_strided(torch.empty(1 << 20, device="cuda", dtype=torch.half), (B, H, s, D), (0, 0, D, 1)) for s in (S, Skv or S))
        return ops.attention_key_scores_workspace_bytes(q, k, k, q, 0.1, causal, noise)
    assert need(1, 71, 300, 64) > 0 and need(1, 71, 299, 64) == 0 and need(1, 16, 600, 64) == 0 and need(1, 16, 700, 64) > 0
    assert need(1, 8, 1000, 128, noise=2) > 0 and need(1, 8, 1000, 128, noise=3) == 0 and need(1, 32, 1501, 128, noise=2) == 0 and need(1, 32, 1501, 128, noise=3) > 0
    assert need(1, 32, 300, 128) > 0 and need(1, 8, 600, 128) == 0 and need(1, 8, 800, 128) > 0 and need(1, 32, 3000, 128) > 0
    assert need(1, 32, 4096, 128) == 0 and need(1, 71, 600, 64, causal=False) == 0 and need(1, 71, 600, 64, Skv=700) == 0
    assert need(64, 71, 128, 64) == 0 and need(1, 71, 4900, 64) == 0
    # few heads with little more than one strip a CU; the longest rows; fp16 noise of long rows; K scattered over the XCDs
    assert need(1, 9, 1001, 64) == 0 and need(1, 8, 1001, 64) > 0 and need(1, 9, 1100, 64) > 0 and need(1, 12, 4600, 64) == 0 and need(1, 8, 4600, 64) > 0
    assert need(1, 8, 4200, 128, noise=2) > 0 and need(1, 8, 4201, 128) == 0 and need(2, 8, 2000, 128, noise=2) > 0 and need(2, 8, 2200, 128, noise=2) == 0
    assert need(1, 24, 1250, 64, noise=2) > 0 and need(1, 24, 1251, 64, noise=2) == 0 and need(1, 24, 1251, 64, noise=3) > 0 and need(1, 16, 2000, 64, noise=2) > 0
    assert need(1, 16, 2500, 128, noise=3) > 0 and need(1, 16, 2700, 128, noise=3) == 0 and need(1, 24, 2700, 128, noise=3) > 0
    assert need(1, 142, 1501, 64, noise=2) == 0 and need(1, 144, 1501, 64, noise=2) > 0 and need(1, 142, 900, 128, noise=3) == 0 and need(1, 142, 700, 128, noise=3) > 0
    q, k, v, n = problem(1, 71, 1, 608, 64, False, 0, 0)
    c, o = torch.empty(1, 71, 608, device="cuda"), torch.empty_like(q)
    m = modules.get("keyformer")
    t = dict(Q=q, K=k, V=v, O=o, noise=n, C_out=c)
    args = [t[p] for p in m.TENSOR_PARAMS]
    m.forward(*args)
    want_c, want_o = c.clone(), o.clone()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        m.forward(*args)
    for _ in range(3):
        c.fill_(-1.0); o.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(c, want_c) and torch.equal(o, want_o)


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("first,later", [(43.0, 43.0), (-43.0, -43.0), (-43.0, 43.0), (43.0, -43.0), (-46.0, 46.0), (60.0, -60.0), (-90.0, 90.0)])
def test_rows_without_a_reference(first, later, half):
    """Scores within 64 of zero, in the log2 domain (44.4), need no reference: rows on both sides of that line, whose first keys and
    whose later ones lie on the same side of zero or on different ones, next to ordinary rows.  In fp16 noise of 32 and more is rounded to 2^-5, which is its value."""
    q, k, v, n = problem(1, 71, 1, 641, 64, half, 0, 0, seed=3)
    n[:, :, 1::3, :256] += first
    n[:, :, 1::3, 256:] += later
    n[:, :, 2::7] += first
    _, rows, c = scores(q, k, v, n, 1.0)
    check(q, k, n, rows, c, 1.0, 5e-5, [(0, 0), (0, 35), (0, 70)], largest=max(abs(first), abs(later)) * 2)


# short prompts and the longest of fp16 noise, at the rule's lines: B, Hq, Hkv, S, D, fp16 noise, spare elements per row, first element
SHORT = [
    (1, 18, 2, 200, 64, False, 1, 0), (1, 20, 4, 201, 64, True, 0, 1), (2, 32, 8, 223, 64, True, 3, 0), (2, 64, 8, 225, 64, False, 0, 0), (2, 71, 1, 380, 64, True, 0, 1),
    (1, 18, 2, 180, 128, False, 0, 1), (1, 40, 8, 180, 128, True, 1, 0), (2, 32, 8, 160, 128, False, 0, 0), (3, 24, 6, 193, 128, False, 3, 1), (2, 40, 8, 255, 128, True, 0, 0),
    (2, 5, 5, 400, 128, False, 0, 0), (1, 48, 8, 1399, 128, True, 1, 0), (1, 32, 8, 1503, 64, True, 0, 0), (4, 71, 1, 200, 64, False, 0, 1),
]
# strips that are no multiple of a head's workgroups: missing from the first round (of one workgroup a CU and of two, an odd and an even number of
# rounds), and from the last
DEALT = [
    (1, 8, 2, 2170, 64, False, 0, 0), (1, 24, 6, 1390, 64, False, 1, 0), (1, 32, 8, 514, 128, False, 0, 0), (1, 44, 4, 743, 64, True, 0, 1), (1, 71, 1, 505, 64, False, 0, 0),
    (1, 71, 1, 820, 128, False, 3, 0), (4, 16, 16, 613, 64, True, 0, 0), (3, 48, 8, 400, 128, False, 0, 1),
]


@pytest.mark.parametrize("B,Hq,Hkv,S,D,half,spare,first", SHORT + DEALT)
def test_one_pass_where_the_rule_begins_and_strips_are_missing(B, Hq, Hkv, S, D, half, spare, first):
    tau, one = 1.5, B * Hq > 240
    q, k, v, n = problem(B, Hq, Hkv, S, D, half, spare, first)
    o, rows, c = scores(q, k, v, n, tau, one_workgroup=one)
    heads = [(0, 0), (B - 1, Hq - 1), (B // 2, Hq // 2)]
    check(q, k, n, rows, c, tau, 2e-5, heads)
    check_outputs(q, k, v, o, heads)


# B, Hq, Hkv, S, D, fp16 noise, one pass: few heads of 128 whose rows are long; three workgroups a head that the chip does not take at once; KV heads that
# the XCDs do not share evenly; fp16 noise of long rows
@pytest.mark.parametrize("B,Hq,Hkv,S,D,half,one_pass", [
    (1, 18, 9, 3401, 128, False, True), (1, 20, 10, 3900, 128, False, True), (1, 28, 14, 3461, 128, False, True), (1, 28, 14, 3500, 128, False, False),
    (1, 30, 15, 3400, 128, False, True), (1, 30, 15, 3401, 128, False, False), (1, 32, 8, 3800, 128, False, True), (1, 32, 8, 3801, 128, False, False),
    (6, 32, 8, 256, 64, False, False), (6, 32, 8, 257, 64, False, True), (5, 34, 2, 200, 64, False, True), (8, 32, 8, 200, 64, False, True), (3, 57, 3, 200, 64, False, False),
    (6, 32, 8, 416, 64, True, True), (6, 32, 8, 417, 64, True, False), (6, 32, 8, 512, 64, True, False), (6, 32, 8, 513, 64, True, True), (5, 41, 1, 450, 64, True, True),
    (6, 32, 8, 560, 128, True, False), (6, 32, 8, 561, 128, True, True), (5, 34, 2, 420, 128, True, True), (5, 41, 1, 420, 128, True, True),
    (1, 96, 24, 1400, 128, True, True), (1, 96, 24, 1401, 128, True, False), (4, 32, 8, 1600, 128, True, True), (4, 32, 8, 1601, 128, True, False),
    (1, 100, 25, 1200, 128, True, True), (1, 100, 25, 1201, 128, True, False), (1, 96, 16, 1400, 128, True, True), (1, 71, 71, 900, 128, True, True), (1, 71, 71, 901, 128, True, False),
    (2, 71, 71, 500, 128, True, False), (1, 100, 25, 1830, 128, False, True), (1, 100, 25, 1840, 128, False, False), (1, 96, 24, 1900, 128, False, True),
])
def test_where_the_single_pass_is_the_faster(B, Hq, Hkv, S, D, half, one_pass):
    from triton_amd import ops
    room = torch.empty(1 << 20, device="cuda", dtype=torch.half)
    q, k = (torch.as_strided(room, (B, H, S, D), (0, 0, D, 1)) for H in (Hq, Hkv))
    # (no size here has one workgroup a head, which needs no workspace)
    assert (ops.attention_key_scores_workspace_bytes(q, k, k, q, 0.1, True, 2 if half else 3) > 0) == one_pass


@pytest.mark.parametrize("B,Hq,Hkv,S,D,half", [(1, 20, 10, 3403, 128, False), (5, 41, 1, 450, 64, True), (6, 32, 8, 561, 128, True)])
def test_one_pass_at_these_lines(B, Hq, Hkv, S, D, half):
    test_one_pass_where_the_rule_begins_and_strips_are_missing(B, Hq, Hkv, S, D, half, 0, 0)


# B, Hq, Hkv, S, fp16 noise, one pass, all of head_dim 128: places that stay empty, KV heads that the XCDs do not share evenly, keys of their own
@pytest.mark.parametrize("B,Hq,Hkv,S,half,one_pass", [
    (4, 66, 6, 496, True, False), (7, 48, 4, 534, True, True), (5, 81, 9, 638, True, False), (7, 27, 9, 941, True, False), (2, 84, 84, 538, True, True), (2, 84, 84, 1001, True, False),
    (2, 66, 66, 538, True, False), (1, 77, 77, 780, True, True), (1, 77, 77, 781, True, False), (1, 95, 95, 560, True, True), (1, 95, 95, 561, True, False),
    (1, 39, 39, 2900, False, True), (1, 39, 39, 3100, False, False), (1, 56, 56, 2500, False, True), (1, 56, 56, 2501, False, False),
])
def test_where_two_passes_are_the_faster(B, Hq, Hkv, S, half, one_pass):
    test_where_the_single_pass_is_the_faster(B, Hq, Hkv, S, 128, half, one_pass)


@pytest.mark.parametrize("B,Hq,Hkv,S,D,half", [(4, 51, 3, 650, 128, True), (1, 95, 95, 545, 128, True)])
def test_one_pass_of_many_heads(B, Hq, Hkv, S, D, half):
    test_one_pass_where_the_rule_begins_and_strips_are_missing(B, Hq, Hkv, S, D, half, 0, 0)
