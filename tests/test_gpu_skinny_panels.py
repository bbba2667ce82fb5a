"""GPU parity of the few-token projections in panels of 32 columns (and of 64 above 128 of those): partial panels, panel counts
around the groups of sixteen that are dealt to the XCDs, matrices that start anywhere among them, k-tiles cut short.

Tolerance: fp16 operands with fp32 accumulation and one rounding to fp16 (2^-11), on outputs of unit variance: 2e-3 of an
output's 2-norm, an element within 2e-3 of itself and 2e-4 of a unit (the fp32 sums' order is far below both).  With an addend
the product is rounded to fp16 before: where that rounding is a tie to the last bits of the fp32 sums it may fall the other way,
one unit in the last place of the product, 2^-10 of it."""
import pytest
import torch

from oracle import ref

pytestmark = pytest.mark.gpu


def close(got, want, product=None):
    d = (got.double() - want).abs()
    off = 2e-4 if product is None else 2e-4 + product.abs() * 2.0 ** -10
    return d.norm() <= 2e-3 * want.norm() and (d <= 2e-3 * want.abs() + off).all()


@pytest.mark.parametrize("T", [1, 15, 16, 17, 24, 25, 32])
@pytest.mark.parametrize("K,cols", [(8, (8,)), (64, (40, 24)), (264, (480, 8, 32)), (520, (520, 512)), (1000, (136, 1000, 24)),
                                    (96, (8192,)), (96, (8200,)), (328, (4096, 2080, 2016))])
def test_linear_panels(T, K, cols):
    from triton_amd import ops
    g = torch.Generator().manual_seed(T * 1000 + K)
    x = ref.randn_half((T, K), g).cuda()
    ws = [ref.randn_half((K, n), g, 0.0, K ** -0.5).cuda() for n in cols]
    add = [ref.randn_half((T, n), g).cuda() if i == 0 else None for i, n in enumerate(cols)]
    outs = [torch.full((T, n), 9.0, dtype=torch.half, device="cuda") for n in cols]
    ops.linear(x, ws, outs)
    for w, o in zip(ws, outs):
        assert close(o, x.double() @ w.double())
    ops.linear(x, ws[:1], outs[:1], add[:1])
    product = (x.double() @ ws[0].double()).half().double()
    assert close(outs[0], product + add[0].double(), product)


@pytest.mark.parametrize("T", [33, 48, 49, 63, 64, 65])
@pytest.mark.parametrize("K,cols", [(8, (8,)), (264, (480, 8, 32)), (1000, (136, 1000, 24)), (96, (8200,))])
def test_linear_panels_of_two_token_blocks(T, K, cols):
    test_linear_panels(T, K, cols)


# 64 MB of weights and more: read past the caches, up to 32 tokens and by the tilings of one tile of tokens
@pytest.mark.parametrize("T,K,cols", [(16, 4104, (8200,)), (32, 4096, (4096, 4096, 40)), (64, 4096, (8200,)), (100, 4096, (8192, 64))])
def test_large_weights(T, K, cols):
    test_linear_panels(T, K, cols)


@pytest.mark.parametrize("T,K,nq,nkv,D,gamma", [(1, 256, 256, 64, 64, True), (16, 1024, 1024, 1024, 64, False), (17, 512, 384, 128, 128, True),
                                                (32, 1032, 1024, 256, 128, True), (24, 328, 64, 64, 64, False),
                                                (50, 512, 512, 128, 128, True), (64, 1032, 1024, 1024, 64, False)])
def test_normalised_projection_panels(T, K, nq, nkv, D, gamma):
    from triton_amd import ops
    g = torch.Generator().manual_seed(K + T)
    x = ref.randn_half((T, K), g, 0.0, 3.0).cuda()
    w = [ref.randn_half((K, n), g, 0.0, K ** -0.5).cuda() for n in (nq, nkv, nkv)]
    gm = ref.randn_half((K,), g, 1.0, 0.1).cuda() if gamma else None
    out = [torch.full((n // D, T, D), 9.0, dtype=torch.half, device="cuda") for n in (nq, nkv, nkv)]
    ops.prenorm_qkv(x, gm, *w, *out, 1e-5, True)
    xd = x.double()
    xn = xd / (xd.pow(2).mean(1, keepdim=True) + 1e-5).sqrt()
    if gamma:
        xn = xn * gm.double()
    for wi, o in zip(w, out):
        # (gamma x is rounded to fp16 before the product: another 2^-11 an operand, the sum of K of them some 3e-4 of the output)
        want = (xn @ wi.double()).view(T, -1, D).permute(1, 0, 2)
        assert (o.double() - want).norm() <= 2e-3 * want.norm() and (o.double() - want).abs().max() <= 4e-3 * want.abs().max()
