"""GPU parity: trn_prenorm_qkv_f16 (fused RMSNorm + QKV GEMM) and the whole PreNorm block against the oracle.
Projections are fp16 outputs of a K=hidden fp32-accumulated GEMM: atol 2e-2 / rtol 1e-2."""
import pytest
import torch

from oracle import ref

pytestmark = pytest.mark.gpu


def close(got, want, atol=2e-2, rtol=1e-2):
    got = got.float().cpu(); want = want.float()
    err = (got - want).abs()
    bad = err > atol + rtol * want.abs()
    assert not bad.any(), f"{int(bad.sum())} off; max abs err {err.max():.4g}"


def weights(g, K, nq, nkv, std=0.02):
    return (ref.randn_half((K, nq), g, 0, std), ref.randn_half((K, nkv), g, 0, std), ref.randn_half((K, nkv), g, 0, std))


@pytest.mark.parametrize("T,K,nq,nkv,D,norm", [(256, 512, 512, 128, 128, True), (130, 520, 192, 64, 64, True),
                                              (16, 4096, 4096, 4096, 128, False), (2048, 4096, 4096, 1024, 128, True),
                                              (1, 64, 64, 64, 64, True), (16, 4544, 4544, 64, 64, True),
                                              # the wide tilings (>= 128 tiles of 256 x 256): ragged tokens and hidden, a
                                              # nearly empty K/V group, no norm -- 256 x 192 tiles (the first three: tiles
                                              # straddle Q | K | V, ragged last tile) and 256 x 256 tiles (the last two)
                                              (1000, 520, 6144, 1024, 128, True), (300, 200, 16384, 64, 64, False),
                                              (900, 264, 8192 + 64, 192, 64, True),
                                              (2048, 200, 6144, 1024, 128, True), (1800, 136, 7168 - 64, 512, 64, False),
                                              # at most 32 tokens: the weight-streaming tiling (four waves split hidden)
                                              (32, 520, 1024, 256, 128, True), (5, 72, 192, 64, 64, True),
                                              (17, 8192, 256, 128, 128, True), (33, 520, 256, 128, 128, True)])
def test_qkv_projection_parity(T, K, nq, nkv, D, norm):
    from triton_amd import ops
    g = torch.Generator().manual_seed(42)
    x = ref.randn_half((T, K), g)
    gamma = ref.randn_half((K,), g, 1.0, 0.02) if norm else None
    wq, wk, wv = weights(g, K, nq, nkv)
    qo = torch.zeros(T, nq, dtype=torch.float16, device="cuda")
    ko = torch.zeros(nkv // D, T, D, dtype=torch.float16, device="cuda")          # head-major
    vo = torch.zeros(T, nkv, dtype=torch.float16, device="cuda")
    ops.prenorm_qkv(x.cuda(), gamma.cuda() if norm else None, wq.cuda(), wk.cuda(), wv.cuda(),
                    qo.view(T, nq // D, D).permute(1, 0, 2), ko, vo.view(T, nkv // D, D).permute(1, 0, 2), 1e-5, norm)
    torch.cuda.synchronize()
    wantq, wantk, wantv = ref.qkv_project(x[None], gamma, wq, wk, wv, 1e-5, norm)
    close(qo, wantq[0]); close(vo, wantv[0])
    close(ko.permute(1, 0, 2).reshape(T, nkv), wantk[0])


def test_projection_into_kv_cache_rows():
    """Decode-append: K, V projections land in rows P..P+M of the [H, P+M, D] caches (ref_rms.py:72-73)."""
    from triton_amd import ops
    M, N, D, P = 16, 512, 64, 40
    H = N // D
    g = torch.Generator().manual_seed(1)
    X = ref.reference_recipe((M, N), g) * 30
    W = [ref.reference_recipe((N, N), g) * 30 for _ in range(3)]
    Kc = ref.reference_recipe((H, P + M, D), g); Vc = ref.reference_recipe((H, P + M, D), g)
    Kd, Vd = Kc.cuda(), Vc.cuda()
    Qd = torch.zeros(H, M, D, dtype=torch.float16, device="cuda")
    ops.prenorm_qkv(X.cuda(), None, W[0].cuda(), W[1].cuda(), W[2].cuda(), Qd, Kd[:, P:], Vd[:, P:], 0.0, False)
    torch.cuda.synchronize()
    q, k, v = ref._decode_qkv(X, *W, D, False)
    assert torch.equal(Kd[:, :P].cpu(), Kc[:, :P]) and torch.equal(Vd[:, :P].cpu(), Vc[:, :P])
    close(Kd[:, P:], k, atol=1e-3); close(Vd[:, P:], v, atol=1e-3); close(Qd, q, atol=1e-3)


@pytest.mark.parametrize("T,K,nq,nkv,D", [(200, 136, 256, 64, 64),         # 128 x 128 tiling
                                         (20, 136, 320, 64, 64),          # weight-streaming tiling
                                         (520, 136, 10240, 512, 128),      # 256 x 192 tiling, tiles straddling Q | K | V
                                         (2048, 136, 6144, 1024, 128)])    # 256 x 256 tiling
def test_projection_reads_and_writes_stay_inside_its_views(T, K, nq, nkv, D):
    """Operands are padded views cut out of NaN-filled buffers, hidden and tokens are ragged: a tile load that strays
    past a row or the end of a view pulls NaN into the product, a store that strays overwrites the NaN padding."""
    from triton_amd import ops
    g = torch.Generator().manual_seed(7)
    x = ref.randn_half((T, K), g); gamma = ref.randn_half((K,), g, 1.0, 0.02)
    wq, wk, wv = weights(g, K, nq, nkv)
    nan = float("nan")

    def padded(t, pad):
        buf = torch.full((t.shape[0] + 3, t.shape[1] + pad), nan, dtype=torch.float16, device="cuda")
        buf[1:1 + t.shape[0], :t.shape[1]] = t.cuda()
        return buf, buf[1:1 + t.shape[0], :t.shape[1]]

    (_, xd), (_, wqd), (_, wkd), (_, wvd) = padded(x, 8), padded(wq, 16), padded(wk, 8), padded(wv, 24)
    outs = []
    for n in (nq, nkv, nkv):
        buf = torch.full((T + 2, n + 8), nan, dtype=torch.float16, device="cuda")
        outs.append((buf, buf[1:1 + T, :n]))
    views = [o[1].unflatten(1, (n // D, D)).permute(1, 0, 2) for o, n in zip(outs, (nq, nkv, nkv))]
    ops.prenorm_qkv(xd, gamma.cuda(), wqd, wkd, wvd, views[0], views[1], views[2], 1e-5, True)
    torch.cuda.synchronize()
    want = ref.qkv_project(x[None], gamma, wq, wk, wv, 1e-5, True)
    for (buf, view), w in zip(outs, want):
        close(view, w[0])
        assert torch.isnan(buf[0]).all() and torch.isnan(buf[T + 1]).all() and torch.isnan(buf[:, view.shape[1]:]).all()


# tokens, hidden, columns of Q and of K and V, head_dim, and the tile that the launcher's rule picks: 64 x 64 tiles up to
# 256 of them, 128 x 64 and then 128 x 128 likewise, two 128 x 128 per CU beyond
@pytest.mark.parametrize("T,K,nq,nkv,D", [(33, 64, 64, 64, 64), (64, 200, 128, 64, 64), (65, 328, 192, 128, 64),       # 64 x 64
                                         (100, 1024, 4096, 1024, 128), (128, 8, 72, 8, 8),
                                         (190, 136, 5504, 256, 128), (256, 264, 6144, 1024, 128),                   # 128 x 64
                                         (385, 136, 6144, 1024, 128), (512, 72, 6144, 1024, 128),                   # 128 x 128
                                         (700, 72, 6144, 1024, 128)])                                               # two per CU
@pytest.mark.parametrize("norm", [False, "plain", "gamma"])
def test_projection_tilings_between_decode_and_long_prompts(T, K, nq, nkv, D, norm):
    """Edges of each tile (tokens, columns, ragged hidden, fewer k-tiles than ring stages) with operands cut out of
    NaN-filled buffers and outputs checked for strays.  Tolerance: one fp16 rounding of the output and, with gamma, one of
    each product gamma * x: 3.6e-4 of the output's spread measured and expected, so 8e-3 of it is more than 20 sigma."""
    from triton_amd import ops
    g = torch.Generator().manual_seed(T + K)
    nan = float("nan")
    x, ws = ref.randn_half((T, K), g), weights(g, K, nq, nkv, K ** -0.5)
    gamma = ref.randn_half((K,), g, 1.0, 0.02) if norm == "gamma" else None

    def padded(t):
        b = torch.full((t.shape[0] + 2, t.shape[1] + 16), nan, dtype=torch.float16, device="cuda")
        b[1:-1, 8:-8] = t.cuda()
        return b[1:-1, 8:-8]
    bufs = [torch.full((T + 2, n + 16), nan, dtype=torch.float16, device="cuda") for n in (nq, nkv, nkv)]
    outs = [b[1:-1, 8:-8].unflatten(1, (n // D, D)).permute(1, 0, 2) for b, n in zip(bufs, (nq, nkv, nkv))]
    ops.prenorm_qkv(padded(x), gamma.cuda() if gamma is not None else None, *[padded(w) for w in ws], *outs, 1e-5, bool(norm))
    torch.cuda.synchronize()
    one = torch.ones(K, dtype=torch.float16)
    want = ref.qkv_project(x[None], gamma if gamma is not None else one, *ws, 1e-5, bool(norm))
    for b, w in zip(bufs, want):
        close(b[1:-1, 8:-8], w[0], atol=8e-3 * float(w.float().std()), rtol=1e-3)
        b[1:-1, 8:-8] = nan
        assert torch.isnan(b).all(), "written outside the output"


@pytest.mark.parametrize("T", [1, 16, 17, 24, 25, 32])
@pytest.mark.parametrize("K", [8, 64, 264, 1000])
def test_weight_stream_at_token_and_hidden_edges(T, K):
    """The three token groups of the decode tiling and contractions from less than one k-tile to several turns of the
    eight waves, norm with gamma, ragged panels; tolerance as above."""
    from triton_amd import ops
    g = torch.Generator().manual_seed(T * K)
    x, gamma = ref.randn_half((T, K), g), ref.randn_half((K,), g, 1.0, 0.02)
    ws = weights(g, K, 200, 72, K ** -0.5)
    outs = [torch.zeros(T, n, dtype=torch.float16, device="cuda") for n in (200, 72, 72)]
    ops.prenorm_qkv(x.cuda(), gamma.cuda(), *[w.cuda() for w in ws],
                    *[o.unflatten(1, (-1, 8)).permute(1, 0, 2) for o in outs], 1e-5, True)
    torch.cuda.synchronize()
    for o, w in zip(outs, ref.qkv_project(x[None], gamma, *ws, 1e-5, True)):
        close(o, w[0], atol=8e-3 * float(w.float().std()), rtol=1e-3)


@pytest.mark.parametrize("T,nq,nkv", [(20, 1024, 256), (64, 1024, 256), (256, 6144, 1024), (512, 6144, 1024), (700, 6144, 1024)])
def test_small_gamma_loses_no_precision(T, nq, nkv):
    """Norm weights around 1e-3 on weights of standard deviation 0.02, every tiling up to two 128 x 128 tiles per CU: the
    products gamma * x stay normal fp16 numbers where gamma * w would not.  One rounding of each product and one of the output,
    2^-11 / sqrt(3) relative at most in the root mean square: 4.0e-4 together (2.9e-4 measured; 8.6e-4 with gamma * w)."""
    from triton_amd import ops
    K = 1024
    g = torch.Generator(device="cuda").manual_seed(T)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x, gamma = r(T, K).half(), (1e-3 * (1 + 0.02 * r(K))).half()
    ws = [(0.02 * r(K, n)).half() for n in (nq, nkv, nkv)]
    outs = [torch.zeros(T, n, dtype=torch.float16, device="cuda") for n in (nq, nkv, nkv)]
    ops.prenorm_qkv(x, gamma, *ws, *[o.unflatten(1, (-1, 64)).permute(1, 0, 2) for o in outs], 1e-5, True)
    torch.cuda.synchronize()
    xd = x.double()
    xn = xd * torch.rsqrt(xd.square().mean(-1, keepdim=True) + 1e-5) * gamma.double()
    for o, w in zip(outs, ws):
        want = xn @ w.double()
        err = float((o.double() - want).norm() / want.norm())
        assert err <= 4.0e-4, err
