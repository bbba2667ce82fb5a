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


@pytest.mark.parametrize("what", ["five axes", "flat output", "two-axis output of other rows"])
def test_rmsnorm_of_any_shape_that_flattens(what):
    """X and X_norm are read as rows of X's last axis, whatever their shapes."""
    from triton_amd import modules
    mod = modules.get("rms")
    a = _tensors(mod)
    want = {n: t.clone() for n, t in a.items()}
    mod.forward(*want.values())
    n = a["X"].numel()
    if what == "five axes":
        a["X"], a["X_norm"] = a["X"].view(2, 1, 3, 2, 256), a["X_norm"].view(2, 1, 3, 2, 256)
    elif what == "flat output":
        a["X_norm"] = a["X_norm"].view(n)
    else:
        a["X_norm"] = a["X_norm"].view(n // 64, 64)
    mod.forward(*a.values())
    torch.cuda.synchronize()
    assert torch.equal(a["X_norm"].view(-1, 256), want["X_norm"])


def test_scores_of_any_contiguous_shape():
    from triton_amd import modules
    mod = modules.get("roco")
    a = _tensors(mod)
    want = {n: t.clone() for n, t in a.items()}
    mod.forward(*want.values())
    a["C_out1"] = a["C_out1"].view(1, 1, 2, 2, 70)
    mod.forward(*a.values())
    torch.cuda.synchronize()
    for n in a:
        assert torch.equal(a[n].reshape(want[n].shape), want[n]), n


def test_operators_refuse_five_axes():
    from triton_amd import ops
    x = torch.zeros(1, 1, 1, 4, 64, dtype=torch.float16, device="cuda")
    with pytest.raises(ValueError):
        ops.rmsnorm(x, None, torch.zeros_like(x), 1e-5)


def test_a_module_copies_after_its_first_forward():
    import copy
    import pickle
    from triton_amd import modules
    mod = modules.get("gmlp", "linear")
    a = _tensors(mod)
    mod.forward(*a.values())
    want = a["O"].clone()
    for other in (copy.deepcopy(mod), copy.copy(mod), pickle.loads(pickle.dumps(mod))):
        a["O"].zero_()
        other.forward(*a.values())
        torch.cuda.synchronize()
        assert torch.equal(a["O"], want)


@pytest.mark.parametrize("variant,form,kw", [("keyformer", "prefill", {}), ("keyformer", "decode", dict(head_dim=64))])
@pytest.mark.parametrize("what", ["same row for every query", "rows far apart", "rows too far apart for the statistics"])
def test_noise_that_the_kernels_cannot_address_is_copied(variant, form, kw, what):
    """fp16 noise expanded along the queries, or with rows further apart than 32-bit offsets within a head reach: in both
    launches, or with the spare rows of the statistics only."""
    from triton_amd import modules
    mod = modules.get(variant, form, **kw)
    a = _tensors(mod)
    n = a["noise"]
    if what == "same row for every query":
        a["noise"] = n[..., :1, :].expand(n.shape)
    else:
        pitch = 0x80000000 // (4 * (n.shape[-2] + (64 if "statistics" in what else 0)))
        wide = torch.empty(n.shape[-2] * pitch, dtype=torch.float16, device="cuda")
        a["noise"] = wide.as_strided(n.shape, (*[n.shape[-1]] * (n.dim() - 2), pitch, 1))      # (heads side by side)
        a["noise"].copy_(n)
    b = {m: t if m == "noise" else t.clone() for m, t in a.items()}
    b["noise"] = a["noise"].float().contiguous()
    mod.forward(*a.values())
    mod.forward(*b.values())
    torch.cuda.synchronize()
    for m in a:
        assert torch.equal(a[m].float(), b[m].float()), m


def test_noise_that_the_statistics_refuse_leaves_the_outputs_alone():
    """A problem of two launches whose second does not take the noise is refused before the first."""
    from triton_amd import _lib, ops
    q = torch.zeros(1, 1, 64, 64, dtype=torch.float16, device="cuda")
    pitch = 0x80000000 // (4 * 128)
    noise = torch.zeros(64 * pitch, dtype=torch.float16, device="cuda").as_strided((1, 1, 64, 64), (0, 0, pitch, 1))
    o, rows, score = torch.full_like(q, 7), torch.full((1, 1, 64), 7.0, device="cuda"), torch.full((1, 1, 64), 7.0, device="cuda")
    with pytest.raises(_lib.TrnError):
        ops.attention_key_scores(q, q, q, o, 1.0, False, rows, score, noise=noise)
    torch.cuda.synchronize()
    assert all(bool((t == 7).all()) for t in (o, rows, score))


def test_other_threads_run_while_a_launch_waits(tmp_path):
    """A forward gives up the interpreter lock for its calls into the library, as a ctypes call does.  In a process of its own,
    with the RMSNorm entry point replaced by one that only sleeps, another thread goes on counting meanwhile."""
    import os
    import subprocess
    import sys
    (tmp_path / "slow.c").write_text("#include <unistd.h>\nint trn_rmsnorm_f16(void) { usleep(400000); return 0; }\n")
    slow = str(tmp_path / "slow.so")
    subprocess.run(["gcc", "-shared", "-fPIC", str(tmp_path / "slow.c"), "-o", slow], check=True)
    child = f"""
import ctypes, threading, time
ctypes.CDLL({slow!r}, mode=ctypes.RTLD_GLOBAL)
import torch
from triton_amd import modules
x = torch.zeros(4, 64, dtype=torch.float16, device="cuda")
mod = modules.get("rms")
mod.forward(x, x.clone(), x[0])
y, n, end = x.clone(), 0, False
def count():
    global n
    while not end:
        n += 1
        time.sleep(0.002)
t = threading.Thread(target=count)
t.start()
time.sleep(0.05)
before, start = n, time.perf_counter()
mod.forward(x, y, x[0])
counted, took = n - before, time.perf_counter() - start
end = True
t.join()
print("took", took, "counted", counted)
assert took > 0.3, "the sleeping entry point was not called"
assert counted > 20
"""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", child], cwd=root, capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
