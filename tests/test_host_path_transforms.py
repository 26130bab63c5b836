"""CPU-side checks that the native host path (csrc/sage_torch.cpp) leaves tensors it cannot take memory and sizes of
— fake, symbolic, batched, differentiated by a transform — to the Python functions behind it, and that
no C++ exception crosses the interpreter's frames.  No device: the tensors are fake ones that say they live on one.
Every case runs in one child process, so that an abort shows as a failed test."""
import subprocess
import sys

import pytest

from mojodiffusion_amd import _lib

CHILD = r"""
import sys
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.fx.experimental.symbolic_shapes import ShapeEnv
from mojodiffusion_amd import _lib, attention_sage as A

h = _lib.host()
case = sys.argv[1]


def calls(t):
    # each entry of the native path; the Python functions ask for the native path first
    g = t[0, 0, 0]
    stats = t[..., :1].float().contiguous()
    return {"fwd": lambda: h.fwd(t, t, t, 0.1, 0, 0, 0, 0, 1), "train": lambda: h.fwd(t, t, t, 0.1, 0, 1, 0, 0, 1),
            "bias": lambda: h.bias(t, t, t, t, 0.1, 0, 1), "norm_rope": lambda: h.norm_rope(t, t, t, g, g, 1e-6, None, None, 0.1, 0, 128, 64, 3, 0, 0),
            "bwd": lambda: h.bwd(t, t, t, t, t, stats, 0.1, 64, 64), "record": lambda: h.record(t, t, t, 0.1, 0)}


def leaves_all(t):
    for name, call in calls(t).items():
        assert call() is None, name


def raises(fn, *args):
    try:
        fn(*args)
    except RuntimeError as e:           # (A.Error is one)
        return str(e)
    raise SystemExit("no error from %s" % fn)


fake = FakeTensorMode(shape_env=ShapeEnv() if case == "symbolic" else None)
with fake:
    t = torch.empty((2, 64, 2, 64), device="cuda", dtype=torch.bfloat16)
if case == "fake":
    leaves_all(t)
    with fake:
        leaves_all(t)
    raises(A.sdpa_nomask, t, t, t, 0.1)
    raises(A.record_sdpa, t, t, t, 0.1)
elif case == "symbolic":
    real = torch.empty((2, 64, 2, 64), dtype=torch.bfloat16)
    from torch._dynamo.source import ConstantSource
    from torch.fx.experimental.symbolic_shapes import DimDynamic, StatelessSymbolicContext
    dyn = StatelessSymbolicContext(dynamic_sizes=[DimDynamic.DYNAMIC] * 4)
    t = fake.from_tensor(real, source=ConstantSource("t"), symbolic_context=dyn)
    with fake:
        t = t.to("cuda")
    assert any(isinstance(n, torch.SymInt) for n in t.shape)
    leaves_all(t)
    raises(A.sdpa_nomask, t, t, t, 0.1)
elif case == "vmap":
    def one(x):
        leaves_all(x)
        leaves_all(t)                   # (a tensor from outside the transform)
        return raises(A.record_sdpa, x, x, x, 0.1) and raises(A.sdpa_nomask, x, x, x, 0.1) and x
    with fake:
        torch.vmap(one)(torch.empty((3, 2, 64, 2, 64), device="cuda", dtype=torch.bfloat16))
elif case == "grad":
    def loss(x):
        leaves_all(x)
        raises(A.sdpa_nomask, x, x, x, 0.1)
        raises(A.record_sdpa, x, x, x, 0.1)
        seen.append(x)
        return x.float().sum()
    seen = []
    try:
        with fake:
            torch.func.grad(loss)(t)
    except RuntimeError:
        assert seen                         # (the engine itself wants a device behind the fake tensors)
elif case == "jvp":
    with fake, torch.autograd.forward_ad.dual_level():
        x = torch.autograd.forward_ad.make_dual(t, torch.ones_like(t))
        leaves_all(x)
elif case == "workspace":
    with fake:
        assert "device memory" in raises(h.workspace, 256, t)       # (a buffer without memory would be handed to every later call)
print("done", case, flush=True)
"""


@pytest.mark.parametrize("case", ["fake", "symbolic", "vmap", "grad", "jvp", "workspace"])
def test_left_to_the_python_path(case):
    r = subprocess.run([sys.executable, "-c", CHILD, case], capture_output=True, text=True, timeout=300, cwd=_lib.os.path.dirname(_lib._HERE))
    assert r.returncode == 0 and r.stdout.split() == ["done", case], (r.returncode, r.stdout[-500:], r.stderr[-1500:])


def test_backward_refuses_a_set_of_another_shape():
    """The kernels take every extent from q and k: a smaller o, d_out, stats or v is refused before its pointer is used."""
    import torch
    from mojodiffusion_amd import attention_sage as A
    q = torch.zeros((1, 64, 2, 64), dtype=torch.bfloat16)
    st = torch.zeros((1, 2, 64, 1))
    half = q[:, :32].contiguous()
    for bad in ({"o": half}, {"d_out": half}, {"v": half}, {"stats": st[:, :, :32]}, {"stats": st.bfloat16()}, {"stats": st.to("meta")}):
        a = {"q": q, "k": q, "v": q, "o": q, "d_out": q, "stats": st, **bad}
        with pytest.raises(A.Error, match="shape|stats|device"):
            A._call_bwd("bwd", *(a[n] for n in ("q", "k", "v", "o", "d_out", "stats")), 0.1, 64, 64)


def test_tables_on_the_host_are_refused():
    """RoPE tables in host memory: an error, not a host pointer in a kernel."""
    import torch
    from torch._subclasses.fake_tensor import FakeTensorMode
    from mojodiffusion_amd import attention_sage as A
    with FakeTensorMode():
        q = torch.empty((1, 64, 2, 64), device="cuda", dtype=torch.bfloat16)
        gain = torch.empty((64,), device="cuda", dtype=torch.bfloat16)
        dev, host = (torch.empty((128, 32), device=d) for d in ("cuda", "cpu"))
        A._norm_rope_args("f", q, q, q, gain, gain, dev, dev)
        for cos, sin in ((host, host), (dev, host), (host, dev)):
            with pytest.raises(A.Error, match="device of q"):
                A._norm_rope_args("f", q, q, q, gain, gain, cos, sin)
