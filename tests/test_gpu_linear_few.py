"""GPU parity of LoRA and the gated MLP of few tokens on little weight, which are one launch each: partial panels, ranks around
the blocks of 32, depths around the turns of eight waves and around the lines between one launch and two, rows at a pitch.

Tolerance: fp16 operands, fp32 sums, every product rounded to fp16 (2^-11 of itself): LoRA's output is the sum of two roundings and its
own, D's roundings reach it through B with unit variance; 2e-3 of the output's 2-norm, 4e-3 for its largest element against the largest."""
import pytest
import torch

from oracle import ref

pytestmark = pytest.mark.gpu


def rows(t, pad):
    """The same values at a row pitch of `pad` elements more, in a buffer of NaNs."""
    b = torch.full((t.shape[0], t.shape[1] + pad), float("nan"), dtype=torch.half, device="cuda")
    b[:, :t.shape[1]] = t
    return b[:, :t.shape[1]]


def close(got, want):
    d = (got.double() - want).abs()
    assert d.norm() <= 2e-3 * want.norm() and d.max() <= 4e-3 * want.abs().max(), f"{d.norm() / want.norm():.2e} {d.max():.2e}"


@pytest.mark.parametrize("T", [1, 15, 16, 17, 32, 33])
@pytest.mark.parametrize("K,P,R,pad", [(8, 8, 8, 0), (40, 40, 24, 8), (1032, 520, 64, 0), (256, 4096, 72, 8), (448, 264, 128, 0), (456, 264, 120, 0),
                                       (1088, 96, 40, 8), (1096, 96, 64, 0), (1448, 1000, 40, 0), (2568, 32, 32, 0), (3592, 32, 24, 0), (264, 4104, 16, 0), (704, 48, 136, 0)])
def test_lora(T, K, P, R, pad):
    from triton_amd import modules
    g = torch.Generator().manual_seed(T + K)
    x, w, a, b = (rows(ref.randn_half(s, g, 0, v).cuda(), pad) for s, v in (((T, K), 1.0), ((K, P), K ** -0.5), ((K, R), K ** -0.5), ((R, P), R ** -0.5)))
    buf = torch.full((T + 2, P + 8), 7.0, dtype=torch.half, device="cuda")
    mod = modules.get("lora", "linear")
    for _ in range(2):
        mod.forward(a, b, buf[1:T + 1, :P], w, x)
    d = (x.double() @ a.double()).half().double()
    close(buf[1:T + 1, :P], x.double() @ w.double() + d @ b.double())
    buf[1:T + 1, :P] = 7.0
    assert (buf == 7.0).all()


@pytest.mark.parametrize("gate", ["sigmoid", "silu"])
@pytest.mark.parametrize("T", [1, 16, 17, 32, 33])
@pytest.mark.parametrize("K,N,pad", [(8, 8, 0), (40, 72, 8), (1024, 1024, 0), (1280, 2056, 0), (1288, 40, 8), (1600, 1032, 0), (1800, 1024, 0), (1808, 64, 0), (264, 4104, 0)])
def test_gated_mlp(T, K, N, pad, gate):
    from triton_amd import modules
    g = torch.Generator().manual_seed(T + K)
    x, w1, w2 = (rows(ref.randn_half(s, g, 0, v).cuda(), pad) for s, v in (((T, K), 1.0), ((K, N), K ** -0.5), ((K, N), K ** -0.5)))
    buf = torch.full((T + 2, N + 8), 7.0, dtype=torch.half, device="cuda")
    modules.get("gmlp", "linear", gate=gate).forward(buf[1:T + 1, :N], w1, w2, x)
    u, v = ((x.double() @ m.double()).half().double() for m in (w1, w2))
    close(buf[1:T + 1, :N], torch.sigmoid(u) * (u if gate == "silu" else 1.0) * v)
    buf[1:T + 1, :N] = 7.0
    assert (buf == 7.0).all()


@pytest.mark.parametrize("T", [5, 20])
def test_no_numbers_stay_in_their_token(T):
    """An infinite activation makes what it makes of two launches, in its own row."""
    from triton_amd import modules, ops
    g = torch.Generator().manual_seed(T)
    K, P, R = 200, 96, 40
    x, w, a, b = (ref.randn_half(s, g, 0, 0.1).cuda() for s in ((T, K), (K, P), (K, R), (R, P)))
    x[3, 7] = float("inf")
    a[7, 5] = 0.0
    o, want, d = (torch.zeros(T, n, dtype=torch.half, device="cuda") for n in (P, P, R))
    modules.get("lora", "linear").forward(a, b, o, w, x)
    ops.linear(x, [w, a], [want, d])
    ops.linear(d, [b], [want], [want])
    assert torch.equal(o.isfinite(), want.isfinite()) and o.isfinite().sum() == (T - 1) * P
    keep = [t for t in range(T) if t != 3]
    close(o[keep], want[keep].double())


@pytest.mark.parametrize("T,K,P,R,pad", [(34, 512, 1000, 16, 0), (64, 1512, 1256, 64, 8), (65, 40, 24, 8, 0), (512, 264, 512, 24, 8), (513, 264, 512, 24, 0), (63, 704, 520, 128, 0),
                                         (70, 328, 2848, 16, 0), (1024, 1000, 504, 32, 8), (1025, 40, 504, 32, 0), (96, 4096, 200, 40, 0), (97, 4104, 200, 40, 0)])
def test_lora_in_tiles_of_tokens(T, K, P, R, pad):
    test_lora(T, K, P, R, pad)


@pytest.mark.parametrize("T,K,N,pad", [(34, 424, 288, 0), (64, 1352, 3024, 8), (65, 8, 8, 0), (512, 384, 416, 8), (513, 384, 416, 0), (95, 4096, 640, 0), (33, 40, 4096, 0), (64, 3072, 40, 0), (64, 3080, 40, 0)])
def test_gated_mlp_in_tiles_of_tokens(T, K, N, pad):
    test_gated_mlp(T, K, N, pad, "silu" if T % 2 else "sigmoid")
