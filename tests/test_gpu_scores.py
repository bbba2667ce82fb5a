"""GPU parity for the key-score paths: forward (row LSE) + trn_attn_colstats_f16, against the CPU oracle.
fp32 key scores: 1e-3 relative.  The absolute allowance is 1e-9: sums of squares of late keys are of order 1e-6 and
below, and a larger allowance would leave exactly those columns unchecked."""
import pytest
import torch

from oracle import ref

pytestmark = pytest.mark.gpu


def close_scores(got, want, rtol=1e-3, atol=1e-9):
    got = got.float().cpu(); want = want.float()
    err = (got - want).abs()
    bad = err > atol + rtol * want.abs()
    assert not bad.any(), f"{int(bad.sum())} off; max rel {(err / want.abs().clamp(min=1e-6)).max():.3g}"


def make(B, Hq, Hkv, Sq, Skv, D, seed=42):
    g = torch.Generator().manual_seed(seed)
    return (ref.randn_half((B, Hq, Sq, D), g), ref.randn_half((B, Hkv, Skv, D), g), ref.randn_half((B, Hkv, Skv, D), g))


def run_roco(q, k, v, scale, causal):
    from triton_amd import ops
    B, Hq, Sq, D = q.shape; Skv = k.shape[2]
    qd, kd, vd = q.cuda(), k.cuda(), v.cuda()
    o = torch.zeros_like(qd); lse = torch.zeros(B, Hq, Sq, device="cuda")
    s1 = torch.full((B, Hq, Skv), -1.0, device="cuda"); s2 = torch.full((B, Hq, Skv), -1.0, device="cuda")
    ops.attention(qd, kd, vd, o, scale, causal, lse=lse)
    ops.attention_colstats(qd, kd, lse, scale, causal, s1, s2)
    torch.cuda.synchronize()
    return o, s1, s2


CASES = [(1, 4, 2, 256, 256, 128, True), (1, 4, 2, 256, 256, 128, False), (2, 3, 1, 200, 200, 64, True),
         (1, 2, 2, 16, 1040, 128, False), (1, 2, 2, 16, 1040, 64, True), (1, 8, 2, 640, 640, 128, True),
         (1, 1, 1, 1, 1, 64, True), (1, 2, 1, 130, 259, 128, True),
         # longer walks of the statistics pass: several mask-free turns of its stage ring, key tiles in pairs with a
         # middle one left over, more queries than keys without a mask, a long cached prefix under the mask
         (1, 1, 1, 1024, 1024, 128, True), (1, 2, 1, 700, 300, 128, False), (1, 2, 2, 520, 1000, 64, True),
         (1, 2, 1, 1100, 1100, 64, True)]


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,D,causal", CASES)
def test_roco_parity(B, Hq, Hkv, Sq, Skv, D, causal):
    q, k, v = make(B, Hq, Hkv, Sq, Skv, D)
    scale = D ** -0.5
    o, s1, s2 = run_roco(q, k, v, scale, causal)
    wo, w1, w2 = ref.roco(q, k, v, scale, causal)
    close_scores(s1, w1); close_scores(s2, w2)
    assert (o.float().cpu() - wo.float()).abs().max() < 2e-2
    # invariant: every row sums to 1, so the column sums add up to the number of queries
    assert torch.allclose(s1.sum(-1).cpu(), torch.full((B, Hq), float(Sq)), rtol=1e-4)


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,D,causal,tau", [
    (1, 4, 2, 256, 256, 128, True, 1.0), (1, 4, 2, 200, 200, 128, True, 1.5), (1, 3, 1, 96, 96, 64, False, 1.0),
    (1, 2, 2, 16, 1040, 128, False, 1.5), (1, 2, 1, 130, 260, 64, True, 1.0),
    (2, 4, 2, 9, 700, 128, True, 1.5), (1, 3, 1, 32, 100, 64, True, 1.0),     # decode kernel with noise, GQA / MQA
    # longer walks of both passes: several turns of the statistics pass's stage ring, a cached prefix, both widths
    (1, 2, 1, 600, 600, 64, True, 1.0), (1, 2, 2, 520, 1000, 128, True, 1.5), (1, 2, 1, 700, 300, 64, False, 1.0)])
def test_keyformer_parity(B, Hq, Hkv, Sq, Skv, D, causal, tau):
    from triton_amd import ops
    q, k, v = make(B, Hq, Hkv, Sq, Skv, D, seed=7)
    noise = ref.gumbel_noise((B, Hq, Sq, Skv), 1234)
    scale = D ** -0.5
    qd, kd, vd, nd = q.cuda(), k.cuda(), v.cuda(), noise.cuda()
    o = torch.zeros_like(qd); lsep = torch.zeros(B, Hq, Sq, device="cuda")
    score = torch.full((B, Hq, Skv), -1.0, device="cuda")
    ops.attention(qd, kd, vd, o, scale, causal, noise=nd, tau=tau, lse_pert=lsep)
    ops.attention_colstats(qd, kd, lsep, scale, causal, score, None, noise=nd, tau=tau)
    torch.cuda.synchronize()
    wo, wscore = ref.keyformer(q, k, v, noise, scale, tau, causal)
    close_scores(score, wscore)
    assert (o.float().cpu() - wo.float()).abs().max() < 2e-2
    assert torch.allclose(score.sum(-1).cpu(), torch.full((B, Hq), float(Sq)), rtol=1e-4)


def _nan_padded(noise):
    """fp32 device copy of `noise` whose rows are padded to a multiple of 4 floats, the padding filled with NaN."""
    B, H, Sq, Skv = noise.shape
    buf = torch.full((B, H, Sq, (Skv + 3) // 4 * 4), float("nan"), device="cuda")
    view = buf[..., :Skv]
    view.copy_(noise)
    return view


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,D,causal,tau", [
    (1, 2, 1, 130, 257, 64, True, 1.0), (1, 2, 2, 203, 203, 128, True, 1.5), (1, 3, 1, 70, 198, 128, False, 1.0),   # prefill kernels
    (1, 4, 2, 16, 1041, 128, False, 1.5), (2, 2, 2, 9, 702, 64, True, 1.0), (1, 3, 1, 32, 99, 128, True, 1.0)])     # decode kernel
def test_keyformer_any_key_count_padding_never_read(B, Hq, Hkv, Sq, Skv, D, causal, tau):
    """The reference's KeyFormer takes any cache length (ref_rms.py:147-179).  The kernels fetch noise 16 bytes at a
    time, so its rows are padded to 4 floats; whatever the padding holds (NaN here) must never reach a sum."""
    from triton_amd import ops
    assert Skv % 4 != 0
    q, k, v = make(B, Hq, Hkv, Sq, Skv, D, seed=21)
    noise = ref.gumbel_noise((B, Hq, Sq, Skv), 77)
    scale = D ** -0.5
    qd, kd, vd, nd = q.cuda(), k.cuda(), v.cuda(), _nan_padded(noise)
    o = torch.zeros_like(qd); lsep = torch.zeros(B, Hq, Sq, device="cuda"); score = torch.full((B, Hq, Skv), -1.0, device="cuda")
    ops.attention_with_stats(qd, kd, vd, o, scale, causal, score, None, noise=nd, tau=tau, lse_pert=lsep)
    torch.cuda.synchronize()
    wo, wscore = ref.keyformer(q, k, v, noise, scale, tau, causal)
    close_scores(score, wscore)
    assert (o.float().cpu() - wo.float()).abs().max() < 2e-2
    s = ref.scores_fp32(q, k, scale, causal)
    assert torch.allclose(lsep.cpu(), torch.logsumexp((s + noise) / tau, -1), atol=1e-3, rtol=1e-3)


def test_keyformer_split_keys_any_key_count():
    from triton_amd import ops
    B, Hq, Hkv, Sq, Skv, D, tau = 1, 8, 2, 16, 4115, 128, 1.5
    q, k, v = make(B, Hq, Hkv, Sq, Skv, D, seed=22)
    noise = ref.gumbel_noise((B, Hq, Sq, Skv), 78)
    scale = D ** -0.5
    qd, kd, vd, nd = q.cuda(), k.cuda(), v.cuda(), _nan_padded(noise)
    o = torch.zeros_like(qd); lse = torch.zeros(B, Hq, Sq, device="cuda"); lsep = torch.zeros_like(lse)
    n = ops.attention_workspace_bytes(qd, kd, vd, o, scale, False)
    assert n > 0
    ws = torch.zeros(n, dtype=torch.uint8, device="cuda")
    ops.attention(qd, kd, vd, o, scale, False, lse=lse, noise=nd, tau=tau, lse_pert=lsep, workspace=ws)
    torch.cuda.synchronize()
    s = ref.scores_fp32(q, k, scale, False)
    assert torch.allclose(lsep.cpu(), torch.logsumexp((s + noise) / tau, -1), atol=1e-3, rtol=1e-3)
    assert (o.float().cpu() - ref.attention(q, k, v, scale, False).float()).abs().max() < 2e-2


@pytest.mark.parametrize("form,PM", [("decode", 1041), ("decode", 1042), ("prefill", 203)])
def test_keyformer_modules_take_fp16_noise_of_any_length(form, PM):
    """Through the module protocol with the reference's fp16 noise (convert_eval_rms.py:201) and a cache length that
    is not a multiple of 4: the module pads its fp32 copy."""
    from triton_amd import modules
    g = torch.Generator().manual_seed(31)
    if form == "decode":
        M, N, D, H = 16, 512, 128, 4
        P = PM - M
        rnd = lambda *sh: (torch.randn(*sh, generator=g).clamp(-1, 1) * 0.05).half()
        X, WQ, WK, WV = rnd(M, N), rnd(N, N), rnd(N, N), rnd(N, N)
        Kc, Vc = rnd(H, PM, D), rnd(H, PM, D)
        noise = torch.randn(H, M, PM, generator=g).half()
        t = dict(X=X.cuda(), WQ=WQ.cuda(), WK=WK.cuda(), WV=WV.cuda(), K_cache=Kc.cuda(), V_cache=Vc.cuda(),
                 O2=torch.zeros(M, N, dtype=torch.float16, device="cuda"), noise=noise.cuda(),
                 C_out=torch.zeros(H, PM, dtype=torch.float16, device="cuda"))
        m = modules.get("keyformer", "decode", head_dim=D)
        m.forward(*[t[p] for p in m.TENSOR_PARAMS])
        torch.cuda.synchronize()
        wo, pw = ref.decode_append_keyformer(X, WQ, WK, WV, Kc, Vc, noise.float(), P, D, tau=1.5)
        assert torch.allclose(t["O2"].float().cpu(), ref.flatten_token_major(wo).float(), atol=2e-2, rtol=1e-2)
        close_scores(t["C_out"], pw.sum(1), rtol=2e-3, atol=1e-3)     # fp16 C_out: its own rounding on top of 1e-3
    else:
        B, Hq, Hkv, S, D = 1, 4, 2, PM, 64
        q, k, v = make(B, Hq, Hkv, S, S, D, seed=32)
        noise = ref.gumbel_noise((B, Hq, S, S), 79).half()
        C_out = torch.zeros(B, Hq, S, device="cuda"); O = torch.zeros(B, Hq, S, D, dtype=torch.float16, device="cuda")
        m = modules.get("keyformer", tau=1.0)
        t = dict(Q=q.cuda(), K=k.cuda(), V=v.cuda(), O=O, noise=noise.cuda(), C_out=C_out)
        m.forward(*[t[p] for p in m.TENSOR_PARAMS])
        torch.cuda.synchronize()
        wo, wc = ref.keyformer(q, k, v, noise.float(), D ** -0.5, 1.0, True)
        close_scores(C_out, wc)
        assert (O.float().cpu() - wo.float()).abs().max() < 2e-2


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,D,causal", [(1, 2, 1, 40, 40, 64, True), (2, 4, 2, 33, 70, 128, True),
                                                      (1, 3, 3, 50, 50, 64, False), (1, 2, 2, 130, 259, 128, True)])
def test_roco_mean_and_std_from_the_kernel_against_numpy(B, Hq, Hkv, Sq, Skv, D, causal):
    """trn_attn_colmeanstd_f16: per-key mean and standard deviation of the probabilities over the queries that see
    the key, held to numpy's mean / std (population) of exactly those entries of the fp64 probability matrix."""
    import numpy as np
    from triton_amd import ops
    q, k, v = make(B, Hq, Hkv, Sq, Skv, D, seed=13)
    scale = D ** -0.5
    qd, kd, vd = q.cuda(), k.cuda(), v.cuda()
    o = torch.zeros_like(qd); lse = torch.zeros(B, Hq, Sq, device="cuda")
    mean = torch.full((B, Hq, Skv), -1.0, device="cuda"); std = torch.full((B, Hq, Skv), -1.0, device="cuda")
    ops.attention(qd, kd, vd, o, scale, causal, lse=lse)
    ops.attention_col_mean_std(qd, kd, lse, scale, causal, mean, std)
    torch.cuda.synchronize()
    p = torch.softmax(ref.scores_fp32(q, k, scale, causal).double(), -1).numpy()
    off = Skv - Sq
    wm = np.zeros((B, Hq, Skv)); ws = np.zeros((B, Hq, Skv))
    for j in range(Skv):
        first = max(0, j - off) if causal else 0              # first query that sees key j
        col = p[:, :, first:, j]
        wm[:, :, j] = col.mean(-1); ws[:, :, j] = col.std(-1)
    close_scores(mean, torch.from_numpy(wm), rtol=1e-3, atol=1e-7)
    # sqrt(E p^2 - mean^2) in fp32 loses digits where the spread is far below the mean; such keys are held to 1e-3
    # of the mean instead
    err = (std.double().cpu() - torch.from_numpy(ws)).abs()
    assert (err <= 2e-3 * torch.from_numpy(ws) + 1e-3 * torch.from_numpy(wm) + 1e-7).all()


def test_uniform_attention_harmonic_closed_form_on_gpu():
    S, D = 300, 128
    q, k, v = make(1, 2, 1, S, S, D, seed=3)
    o, s1, s2 = run_roco(torch.zeros_like(q), k, v, 1.0, True)
    want1 = ref.harmonic_tail(S, 1).float(); want2 = ref.harmonic_tail(S, 2).float()
    close_scores(s1[0, 0], want1, rtol=1e-4); close_scores(s2[0, 1], want2, rtol=1e-4)


def test_colstats_deterministic():
    q, k, v = make(1, 4, 2, 384, 384, 128, seed=5)
    _, a1, a2 = run_roco(q, k, v, 0.088, True)
    _, b1, b2 = run_roco(q, k, v, 0.088, True)
    assert torch.equal(a1, b1) and torch.equal(a2, b2)


# ---- trn_attn_fwd_stats_f16: attention + statistics in one call (one launch with at most 32 queries per head)
FUSED = [(1, 4, 4, 16, 1040, 128, False), (1, 4, 2, 16, 1040, 128, True), (2, 6, 1, 7, 333, 64, True),
         (1, 3, 3, 32, 32, 128, True), (1, 2, 2, 1, 100, 64, False), (1, 71, 1, 16, 1040, 64, False),
         (1, 4, 2, 130, 259, 128, True)]                     # more than 32 queries: two launches inside the call


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,D,causal", FUSED)
def test_fused_attention_and_roco_statistics(B, Hq, Hkv, Sq, Skv, D, causal):
    from triton_amd import ops
    q, k, v = make(B, Hq, Hkv, Sq, Skv, D, seed=11)
    scale = D ** -0.5
    qd, kd, vd = q.cuda(), k.cuda(), v.cuda()
    o = torch.zeros_like(qd); lse = torch.zeros(B, Hq, Sq, device="cuda")
    s1 = torch.full((B, Hq, Skv), -1.0, device="cuda"); s2 = torch.full((B, Hq, Skv), -1.0, device="cuda")
    ops.attention_with_stats(qd, kd, vd, o, scale, causal, s1, s2, lse=lse)
    torch.cuda.synchronize()
    wo, w1, w2 = ref.roco(q, k, v, scale, causal)
    close_scores(s1, w1); close_scores(s2, w2)
    assert (o.float().cpu() - wo.float()).abs().max() < 2e-2
    assert torch.allclose(s1.sum(-1).cpu(), torch.full((B, Hq), float(Sq)), rtol=1e-4)
    # the same numbers as the two separate calls (within summation order)
    o2, t1, t2 = run_roco(q, k, v, scale, causal)
    close_scores(s1, t1.cpu(), rtol=1e-4); close_scores(s2, t2.cpu(), rtol=1e-4)
    # only one of the two statistics
    s1b = torch.full_like(s1, -1.0)
    ops.attention_with_stats(qd, kd, vd, o, scale, causal, s1b, None, lse=lse)
    torch.cuda.synchronize()
    assert torch.equal(s1b, s1)


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,D,causal,tau", [(1, 4, 4, 16, 1040, 128, False, 1.5), (2, 4, 2, 9, 700, 128, True, 1.5),
                                                          (1, 3, 1, 32, 100, 64, True, 1.0), (1, 2, 1, 130, 260, 64, True, 1.0)])
def test_fused_attention_and_keyformer_scores(B, Hq, Hkv, Sq, Skv, D, causal, tau):
    from triton_amd import ops
    q, k, v = make(B, Hq, Hkv, Sq, Skv, D, seed=7)
    noise = ref.gumbel_noise((B, Hq, Sq, Skv), 1234)
    scale = D ** -0.5
    o = torch.zeros_like(q).cuda(); lsep = torch.zeros(B, Hq, Sq, device="cuda")
    score = torch.full((B, Hq, Skv), -1.0, device="cuda")
    ops.attention_with_stats(q.cuda(), k.cuda(), v.cuda(), o, scale, causal, score, None, noise=noise.cuda(), tau=tau, lse_pert=lsep)
    torch.cuda.synchronize()
    wo, wscore = ref.keyformer(q, k, v, noise, scale, tau, causal)
    close_scores(score, wscore)
    assert (o.float().cpu() - wo.float()).abs().max() < 2e-2
    assert torch.allclose(score.sum(-1).cpu(), torch.full((B, Hq), float(Sq)), rtol=1e-4)


def test_fused_statistics_argument_rules():
    from triton_amd import ops, _lib
    q, k, v = make(1, 2, 2, 64, 64, 64)
    qd, kd, vd = q.cuda(), k.cuda(), v.cuda()
    o = torch.zeros_like(qd); s1 = torch.zeros(1, 2, 64, device="cuda")
    with pytest.raises(_lib.TrnError) as e:          # more than 32 queries and no buffer for the row normalisers
        ops.attention_with_stats(qd, kd, vd, o, 0.125, True, s1)
    assert e.value.status_name == "TRN_E_NULL"
    with pytest.raises(ValueError):
        ops.attention_with_stats(qd, kd, vd, o, 0.125, True, None, None)


# ---- trn_attn_fwd_stats_half_f16: the same launch with fp16 noise and fp16 statistics (the reference's own tensors)
@pytest.mark.gpu
@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,D,causal,with_noise", [
    (1, 4, 4, 16, 1040, 128, False, True), (1, 4, 2, 16, 1040, 128, True, False), (2, 6, 1, 7, 332, 64, True, True),
    (1, 71, 1, 16, 1040, 64, False, False), (1, 3, 3, 32, 36, 128, True, True), (1, 2, 2, 1, 100, 64, False, True),
    # odd key counts: the last row's last key sits in a dword that is half padding
    (1, 4, 4, 16, 333, 128, True, True), (1, 2, 1, 16, 1041, 64, False, True), (1, 2, 2, 3, 35, 128, False, True)])
def test_fused_statistics_with_fp16_noise_and_outputs(B, Hq, Hkv, Sq, Skv, D, causal, with_noise):
    """Held to the fp32 form of the same call bit for bit: the fp16 noise widened is the same noise, and an fp16 statistic
    is the fp32 one rounded once.  (The fp32 form is held to the oracle above.)"""
    from triton_amd import ops
    q, k, v = make(B, Hq, Hkv, Sq, Skv, D, seed=17)
    scale, tau = D ** -0.5, 1.5
    qd, kd, vd = q.cuda(), k.cuda(), v.cuda()
    g = torch.Generator().manual_seed(5)
    pitch = (Skv + 3) // 4 * 4
    n16 = torch.full((B, Hq, Sq, pitch), float("nan"), dtype=torch.float16)
    n16[..., :Skv] = torch.randn(B, Hq, Sq, Skv, generator=g).half()
    n16 = n16.cuda()[..., :Skv] if with_noise else None
    n32 = None
    if with_noise:
        buf = torch.full((B, Hq, Sq, pitch), float("nan"), device="cuda"); buf[..., :Skv] = n16.float(); n32 = buf[..., :Skv]
    o1 = torch.zeros_like(qd); o2 = torch.zeros_like(qd)
    lp1 = torch.zeros(B, Hq, Sq, device="cuda"); lp2 = torch.zeros_like(lp1)
    a1 = torch.full((B, Hq, Skv), -1.0, device="cuda"); a2 = torch.full((B, Hq, Skv), -1.0, device="cuda")
    h1 = torch.full((B, Hq, Skv), -1.0, device="cuda", dtype=torch.float16); h2 = torch.full_like(h1, -1.0)
    kw32 = dict(noise=n32, tau=tau, lse_pert=lp1) if with_noise else dict(lse=lp1)
    kw16 = dict(noise=n16, tau=tau, lse_pert=lp2) if with_noise else dict(lse=lp2)
    ops.attention_with_stats(qd, kd, vd, o1, scale, causal, a1, a2, **kw32)
    ops.attention_with_stats_half(qd, kd, vd, o2, scale, causal, h1, h2, **kw16)
    torch.cuda.synchronize()
    assert torch.equal(o1, o2) and torch.equal(lp1, lp2)
    assert torch.equal(h1, a1.half()) and torch.equal(h2, a2.half())


@pytest.mark.gpu
def test_fp16_statistics_form_refuses_prefill_shapes():
    from triton_amd import ops
    q, k, v = make(1, 2, 2, 33, 64, 64)
    qd, kd, vd = q.cuda(), k.cuda(), v.cuda()
    h1 = torch.zeros(1, 2, 64, device="cuda", dtype=torch.float16)
    with pytest.raises(ValueError):
        ops.attention_with_stats_half(qd, kd, vd, torch.zeros_like(qd), 0.125, True, h1)


# ---- trn_attn_key_scores_f16: any noise element type, pitch and alignment, fp16 or fp32 statistics, every kernel behind it
@pytest.mark.gpu
@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,D,causal,ws", [
    (1, 4, 2, 16, 333, 128, True, False), (1, 3, 3, 1, 35, 64, False, False), (1, 8, 2, 16, 8193, 128, False, True),   # decode, split keys
    (2, 4, 2, 65, 129, 128, True, False), (1, 71, 1, 100, 131, 64, False, False),                                      # tiles of 32 queries
    (4, 32, 8, 131, 131, 128, True, False), (2, 71, 1, 150, 217, 64, True, False), (8, 32, 8, 257, 257, 64, True, False)])  # prefill kernels
@pytest.mark.parametrize("noise", ["fp16", "fp32"])
def test_key_scores_for_noise_at_any_pitch(B, Hq, Hkv, Sq, Skv, D, causal, ws, noise):
    """Rows of Skv (odd) elements without padding, the whole tensor starting one element into its buffer: held bit for bit to
    the entry point that takes padded fp32 noise (and that the oracle tests above cover); fp16 statistics are the fp32
    ones rounded once.  The words around the tensor are NaN."""
    from triton_amd import ops
    q, k, v = (t.cuda() for t in make(B, Hq, Hkv, Sq, Skv, D, seed=11))
    dt = torch.float16 if noise == "fp16" else torch.float32
    n = B * Hq * Sq * Skv
    buf = torch.full((n + 9,), float("nan"), dtype=dt, device="cuda")
    x = buf[1:n + 1].view(B, Hq, Sq, Skv)
    x.copy_(torch.randn(B, Hq, Sq, Skv, generator=torch.Generator().manual_seed(2)))
    pad = torch.full((B, Hq, Sq, (Skv + 3) // 4 * 4), float("nan"), device="cuda")
    pad[..., :Skv] = x.float()
    scale, stat = D ** -0.5, lambda dt=torch.float32: torch.full((B, Hq, Skv), -1.0, device="cuda", dtype=dt)
    work = None
    if ws:
        nb = ops.attention_stats_workspace_bytes(q, k, v, q, scale, causal)
        assert nb > 0
        work = torch.zeros(nb, dtype=torch.uint8, device="cuda")
    o1, o2, o3 = torch.zeros_like(q), torch.zeros_like(q), torch.zeros_like(q)
    r1, r2 = torch.zeros(B, Hq, Sq, device="cuda"), torch.zeros(B, Hq, Sq, device="cuda")
    a1, b1, a2, b2 = stat(), stat(), stat(), stat()
    h1, h2 = stat(torch.float16), stat(torch.float16)
    ops.attention_with_stats(q, k, v, o1, scale, causal, a1, b1, noise=pad[..., :Skv], tau=1.5, lse_pert=r1, workspace=work)
    ops.attention_key_scores(q, k, v, o2, scale, causal, r2, a2, b2, noise=x, tau=1.5, workspace=work)
    ops.attention_key_scores(q, k, v, o3, scale, causal, r2, h1, h2, noise=x, tau=1.5, workspace=work)
    torch.cuda.synchronize()
    assert torch.equal(o1, o2) and torch.equal(o1, o3) and torch.equal(r1, r2)
    assert torch.equal(a1, a2) and torch.equal(b1, b2)
    assert torch.equal(h1, a1.half()) and torch.equal(h2, b1.half())


@pytest.mark.gpu
@pytest.mark.parametrize("Sq,Skv", [(16, 100), (200, 200)])
def test_key_scores_without_noise_and_as_mean_and_std(Sq, Skv):
    from triton_amd import ops, _lib
    q, k, v = (t.cuda() for t in make(1, 4, 2, Sq, Skv, 128, seed=12))
    stat = lambda: torch.full((1, 4, Skv), -1.0, device="cuda")
    lse, rows = torch.zeros(1, 4, Sq, device="cuda"), torch.zeros(1, 4, Sq, device="cuda")
    o1, o2, s = torch.zeros_like(q), torch.zeros_like(q), [stat() for _ in range(8)]
    ops.attention(q, k, v, o1, 0.1, True, lse=lse)
    ops.attention_with_stats(q, k, v, o1, 0.1, True, s[0], s[1], lse=lse)
    ops.attention_col_mean_std(q, k, lse, 0.1, True, s[2], s[3])
    ops.attention_key_scores(q, k, v, o2, 0.1, True, rows, s[4], s[5])
    ops.attention_key_scores(q, k, v, o2, 0.1, True, rows, s[6], s[7], mean_std=True)
    torch.cuda.synchronize()
    assert torch.equal(o1, o2) and torch.equal(lse, rows) and all(torch.equal(s[i], s[i + 4]) for i in range(4))
    with pytest.raises(ValueError):
        ops.attention_key_scores(q, k, v, o2, 0.1, True, rows, s[4], s[5].half())
    with pytest.raises(_lib.TrnError):           # mean and standard deviation are defined without noise only
        ops.attention_key_scores(q, k, v, o2, 0.1, True, rows, s[4], s[5], noise=torch.zeros(1, 4, Sq, Skv, device="cuda"), mean_std=True)


# ---- forward kernel with perturbed scores: the mask-free loop and its late raises of the two running references
@pytest.mark.gpu
@pytest.mark.parametrize("Sq,Skv,causal", [(576, 95, False), (577, 96, False), (600, 159, False), (600, 160, False), (600, 225, False),
                                           (513, 513, True), (640, 640, True), (600, 791, True), (1025, 1025, True)])
@pytest.mark.parametrize("Hq,Hkv,D", [(2, 1, 128), (2, 2, 64)])
@pytest.mark.parametrize("noise", ["fp16", "fp32"])
def test_perturbed_scores_that_grow_along_the_keys(Sq, Skv, causal, Hq, Hkv, D, noise):
    """Keys whose scores and noise grow with their index, so that both references are raised in every part of the walk:
    sizes around whole turns of the mask-free loop.  Tolerances as for the other key-score tests (probabilities from fp16
    products, 1e-3), row normalisers 1e-3."""
    from triton_amd import ops
    q, k, v = make(1, Hq, Hkv, Sq, Skv, D, seed=31)
    ramp = torch.arange(Skv, dtype=torch.float32)
    # shifts of a key by up to 12 in the scaled scores: a component of q that is 1 everywhere meets the ramp
    q[..., 0] = 1.0
    k[..., 0] = (12.0 * D ** 0.5 * ramp / Skv).half()
    x = (torch.randn(1, Hq, Sq, Skv, generator=torch.Generator().manual_seed(5)) + 60.0 * ramp / Skv).half()
    nd = x.cuda() if noise == "fp16" else x.float().cuda()
    scale, qd, kd, vd = D ** -0.5, q.cuda(), k.cuda(), v.cuda()
    o, rows = torch.zeros_like(qd), torch.zeros(1, Hq, Sq, device="cuda")
    score = torch.full((1, Hq, Skv), -1.0, device="cuda")
    ops.attention_key_scores(qd, kd, vd, o, scale, causal, rows, score, None, noise=nd, tau=1.0)
    torch.cuda.synchronize()
    wo, wscore = ref.keyformer(q, k, v, x.float(), scale, 1.0, causal)
    close_scores(score, wscore, atol=1e-6)      # (early keys: e^-60 of a row, below fp32's reach of a column sum)
    assert (o.float().cpu() - wo.float()).abs().max() < 2e-2
    s = ref.scores_fp32(q, k, scale, causal)
    assert torch.allclose(rows.cpu(), torch.logsumexp(s + x.float(), -1), atol=1e-3, rtol=1e-3)


# ---- statistics with noise: one and two groups of waves per workgroup, either side of the rule, ragged group ends
@pytest.mark.gpu
@pytest.mark.parametrize("Sq,Skv,causal", [(320, 320, True), (321, 321, True), (385, 130, False), (449, 700, True), (512, 64, False),
                                           (1537, 1537, True), (1025, 1100, True)])
@pytest.mark.parametrize("B,Hq,Hkv,D", [(1, 3, 1, 128), (2, 2, 2, 64), (4, 8, 2, 64)])
@pytest.mark.parametrize("noise", ["fp16", "fp32"])
def test_key_sums_and_squares_by_one_or_two_groups_of_waves(Sq, Skv, causal, B, Hq, Hkv, D, noise):
    """Held to float64 sums over the probabilities that the same row normalisers give: 2e-5 relative covers fp32 scores of
    D products (|score| < 2^4 in the log2 domain: 16 * 2^-24 * sqrt(D) of an exponent) and fp32 sums of 1600 terms."""
    from triton_amd import ops
    q, k, _ = (t.cuda() for t in make(B, Hq, Hkv, Sq, Skv, D, seed=41))
    x = torch.randn(B, Hq, Sq, Skv, generator=torch.Generator(device="cuda").manual_seed(6), device="cuda").half()
    nd = x if noise == "fp16" else x.float()
    scale = D ** -0.5
    s = (q.double() @ k.double().repeat_interleave(Hq // Hkv, 1).transpose(-1, -2).contiguous()) * scale + x.double()
    if causal:
        s = s.masked_fill(~torch.ones(Sq, Skv, dtype=torch.bool, device="cuda").tril(Skv - Sq), float("-inf"))
    o, rows = torch.zeros_like(q), torch.zeros(B, Hq, Sq, device="cuda")
    s1, s2 = (torch.full((B, Hq, Skv), -1.0, device="cuda") for _ in range(2))
    v = torch.zeros_like(k)
    ops.attention_key_scores(q, k, v, o, scale, causal, rows, s1, s2, noise=nd, tau=1.0)
    torch.cuda.synchronize()
    p = torch.exp(s - rows.double().unsqueeze(-1))
    for got, want in ((s1, p.sum(2)), (s2, p.square().sum(2))):
        assert ((got.double() - want).abs() <= 2e-5 * want + 1e-12).all(), ((got.double() - want).abs() / want).max()


# ---- the furthest rows that the statistics kernels can address: their requests past the last query still read zeros
@pytest.mark.gpu
@pytest.mark.parametrize("Sq", [1, 64, 200, 321, 385])
@pytest.mark.parametrize("noise", [None, "fp16", "fp32"])
def test_statistics_at_the_largest_row_pitch(Sq, noise):
    """Query and noise rows as far apart as TRN_STATS_SPARE_ROWS = 128 allows, walks of one and of two groups of waves with
    short last tiles: the bits of compact tensors."""
    from triton_amd import ops
    D, Skv = 64, 130

    def apart(t, elem_bytes):
        pitch = 0x7fffffff // ((Sq + 128) * elem_bytes) // 8 * 8
        w = torch.empty((Sq - 1) * pitch + t.shape[-1], dtype=t.dtype, device="cuda").as_strided(t.shape, (0, 0, pitch, 1))
        return w.copy_(t)
    q, k, v = (t.cuda() for t in make(1, 1, 1, Sq, Skv, D, seed=51))
    n = None if noise is None else torch.randn(1, 1, Sq, Skv, device="cuda").to(torch.float16 if noise == "fp16" else torch.float32)
    got = []
    for wide in (False, True):
        qw, nw = (apart(q, 2), None if n is None else apart(n, 4)) if wide else (q, n)
        o, rows, s1, s2 = torch.zeros_like(q), torch.zeros(1, 1, Sq, device="cuda"), *(torch.zeros(1, 1, Skv, device="cuda") for _ in range(2))
        if Sq > 32:
            ops.attention_key_scores(qw, k, v, o, 0.125, False, rows, s1, s2, noise=nw, tau=1.0)
        elif noise != "fp16":            # (the single launch of a few queries has its own sweep: the statistics alone here)
            ops.attention_colstats(qw, k, rows, 0.125, False, s1, s2, noise=nw if n is None or wide else torch.nn.functional.pad(n, (0, 2))[..., :Skv])
        torch.cuda.synchronize()
        got.append((o, rows, s1, s2))
    assert all(torch.equal(a, b) for a, b in zip(*got))


# ---- a row whose first keys carry a mask: the first reference of the perturbed scores lies far below zero
@pytest.mark.gpu
@pytest.mark.parametrize("Hq,Hkv,D,Sq", [(2, 1, 128, 100), (32, 8, 128, 600), (32, 8, 64, 600)])      # 32-query tiles, prefill kernel
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("first,low", [(40, -200.0), (32, -65504.0), (110, -65504.0)])
def test_noise_that_masks_the_first_keys(Hq, Hkv, D, Sq, dtype, first, low):
    """Keys [0, first) of every row at `low`, under the causal mask: rows before `first` see nothing else.  Scores next to a
    reference of the size of `low` carry its rounding, 2^-24 * |low| / ln 2 of an exponent: 0.4 % for -65504, in the block that a
    row leaves the mask in and, twice, throughout the rows that see nothing else.  Beyond that the 1e-3 of the tests above (2e-3
    for the normalisers)."""
    from triton_amd import ops
    q, k, v = (t.cuda() for t in make(1, Hq, Hkv, Sq, Sq, D, seed=61))
    n = torch.randn(1, Hq, Sq, Sq, generator=torch.Generator(device="cuda").manual_seed(7), device="cuda").to(dtype)
    n[..., :first] = low
    o, rows, score = torch.zeros_like(q), torch.zeros(1, Hq, Sq, device="cuda"), torch.zeros(1, Hq, Sq, device="cuda")
    ops.attention_key_scores(q, k, v, o, D ** -0.5, True, rows, score, noise=n, tau=1.0)
    torch.cuda.synchronize()
    s = q[0].double() @ k[0].double().repeat_interleave(Hq // Hkv, 0).transpose(-1, -2).contiguous() * D ** -0.5 + n[0].double()
    s = s.masked_fill(~torch.ones(Sq, Sq, dtype=torch.bool, device="cuda").tril(), float("-inf"))
    lse, p = torch.logsumexp(s, -1), s.softmax(-1).sum(1)
    spoilt = 2 ** -24 * -low / 0.6931
    assert ((rows[0].double() - lse).abs() <= 2e-3 + spoilt + 2 ** -23 * lse.abs()).all()
    assert ((score[0].double() - p).abs()[:, first:] <= (1e-3 + spoilt) * p[:, first:] + 1e-9).all()
    assert ((score[0].double() - p).abs()[:, :first] <= (1e-3 + 2 * spoilt) * p[:, :first]).all()
