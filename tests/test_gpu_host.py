"""The modules' native forward against their general Python path: same bits for what both cover, and the general path
itself for layouts and types the native one declines."""
import pytest
import torch

from oracle import ref

pytestmark = pytest.mark.gpu


def _tensors(mod, M=12, H=4, D=64, P=50, S=70):
    g = torch.Generator().manual_seed(4)
    N = H * D
    r = lambda *s, std=1.0: ref.randn_half(s, g, 0.0, std).cuda()
    decode = "K_cache" in mod.TENSOR_PARAMS
    t = dict(X=r(M, N), WQ=r(N, N, std=N ** -0.5), WK=r(N, N, std=N ** -0.5), WV=r(N, N, std=N ** -0.5), K_cache=r(H, P + M, D),
             V_cache=r(H, P + M, D), O2=r(M, N), Q=r(1, H, S, D), K=r(1, H // 2, S, D), V=r(1, H // 2, S, D),
             gamma_q=r(D), gamma_k=r(D), gamma=r(N), X_norm=r(M, N), A=r(N, 16, std=0.1), B=r(16, 40, std=0.1), W=r(N, 40, std=0.1),
             W1=r(N, 48, std=0.1), W2=r(N, 48, std=0.1), noise=r(H, M, P + M) if decode else r(1, H, S, S),
             O={"LoRA": r(M, 40), "GatedMLP": r(M, 48), "PreNormBlock": r(M, N)}.get(type(mod).__name__, r(1, H, S, D)))
    for n in ("C_out", "C_out1", "C_out2"):
        t[n] = torch.zeros((H, P + M) if decode else (1, H, S), device="cuda")
    return {n: t[n] for n in mod.TENSOR_PARAMS}


CASES = [("rms", "prefill", {}), ("vanilla", "prefill", {}), ("qknorm", "prefill", {}), ("keyformer", "prefill", {}), ("roco", "prefill", {}),
         ("roco", "prefill", dict(stats="mean_std")), ("prenorm", "prefill", dict(head_dim=64)), ("vanilla", "decode", dict(head_dim=64)),
         ("prenorm", "decode", dict(head_dim=64, causal=True)), ("qknorm", "decode", dict(head_dim=64, o_layout="head_major")),
         ("keyformer", "decode", dict(head_dim=64)), ("roco", "decode", dict(head_dim=64)), ("lora", "linear", {}), ("gmlp", "linear", dict(gate="silu"))]


@pytest.mark.parametrize("variant,form,kw", CASES)
def test_native_forward_equals_the_general_path(variant, form, kw):
    from triton_amd import modules
    mod = modules.get(variant, form, **kw)
    a = _tensors(mod)
    b = {n: t.clone() for n, t in a.items()}
    mod.forward(*a.values())
    assert mod._native(mod._host, mod._hws, *a.values()) is True, "expected the native path to take these tensors"
    mod._run(*b.values())
    torch.cuda.synchronize()
    for n in a:
        assert torch.equal(a[n], b[n]), n


@pytest.mark.parametrize("what", ["mixed statistics", "strided statistics", "fp64 noise", "three-axis strided X"])
def test_layouts_the_native_forward_declines_still_run(what):
    from triton_amd import modules
    mod = modules.get(*{"mixed statistics": ("roco", "decode"), "strided statistics": ("roco", "decode"), "fp64 noise": ("keyformer", "decode"),
                        "three-axis strided X": ("rms", "prefill")}[what], **({} if "X" in what else dict(head_dim=64)))
    a = _tensors(mod)
    want = {n: t.clone() for n, t in a.items()}
    mod.forward(*want.values())
    if what == "mixed statistics":
        a["C_out1"] = a["C_out1"].half()
    elif what == "strided statistics":
        a["C_out2"] = torch.zeros(*a["C_out2"].shape, 2, device="cuda")[..., 0]
    elif what == "fp64 noise":
        a["noise"] = a["noise"].double()
    else:
        x = torch.zeros(3, 4, 512, dtype=torch.float16, device="cuda")[..., :256]
        x.copy_(a["X"].view(3, 4, 256)); a["X"] = x
        y = torch.zeros(3, 4, 512, dtype=torch.float16, device="cuda")[..., :256]
        a["X_norm"] = y
    mod.forward(*a.values())
    torch.cuda.synchronize()
    for n in a:
        if n in ("X",):
            continue
        assert torch.equal(a[n].to(want[n].dtype).reshape(want[n].shape) if n != "C_out1" else a[n].float(),
                           want[n] if n != "C_out1" or what != "mixed statistics" else want[n].half().float()), n
