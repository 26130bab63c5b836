"""GPU tests of the native host path (csrc/sage_torch.cpp) and of what it calls besides the entry points tested
elsewhere: the boundary casts, the bias with rows at any start, the recorded node.  The Python path behind it is
the reference: same kernels, so the same bits."""
import ctypes

import numpy as np
import pytest

from mojodiffusion_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(1,), (7, 8, 9), (2047, 2048, 2049, 100003)])
def test_casts_round_like_torch(sizes):
    """F32 -> bf16 to nearest even (ties, infinities, subnormals; NaN stays NaN) and back, tensors of any length."""
    import torch
    L = _lib.lib()
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    src = [torch.randn(n, device="cuda", generator=g) * 10.0 ** float(i * 12 - 20) for i, n in enumerate(sizes)]
    special = torch.tensor([1.00390625, 1.01171875, -1.00390625, float("inf"), -float("inf"), float("nan"), 1e-40, -0.0], device="cuda")
    src[-1][:min(8, src[-1].numel())] = special[:min(8, src[-1].numel())]
    dst = [torch.full((t.numel() + 1,), 7.0, device="cuda").bfloat16() for t in src]
    back = [torch.full((t.numel() + 1,), 7.0, device="cuda") for t in src]
    n = len(src)
    ptrs = lambda ts: (ctypes.c_void_p * n)(*(t.data_ptr() for t in ts))
    lens = (ctypes.c_int64 * n)(*sizes)
    st = torch.cuda.current_stream().cuda_stream
    assert L.mi355_sage_cast(n, ptrs(src), ptrs(dst), lens, 1, st) == 0
    assert L.mi355_sage_cast(n, ptrs(dst), ptrs(back), lens, 0, st) == 0
    torch.cuda.synchronize()
    for s, d, b in zip(src, dst, back):
        want, k = s.bfloat16(), s.numel()
        assert torch.equal(torch.isnan(d[:k]), torch.isnan(want)) and torch.equal(d[:k].nan_to_num(5.0), want.nan_to_num(5.0))
        assert torch.equal(b[:k].nan_to_num(5.0), want.float().nan_to_num(5.0))
        assert float(d[k]) == 7.0 and float(b[k]) == 7.0                    # nothing past the end
    assert L.mi355_sage_cast(5, ptrs(src), ptrs(dst), lens, 1, st) == -1


@pytest.mark.parametrize("variant,Sq,Skv,D", [(0, 70, 77, 128), (1, 33, 129, 64), (0, 600, 1031, 128), (0, 40, 6, 256)])
def test_bias_rows_at_any_start(variant, Sq, Skv, D):
    """A contiguous bias of odd key count: the bits of the same bias in rows padded to four keys."""
    import torch
    from mojodiffusion_amd import attention_sage as A
    torch.manual_seed(Sq)
    q, k, v = (torch.randn((2, n, 3, D), device="cuda").bfloat16() for n in (Sq, Skv, Skv))
    bias = torch.randn((2, 3, Sq, Skv), device="cuda").bfloat16()
    got = A.sdpa_cross_masked(q, k, v, bias, D ** -0.5, variant)
    padded = torch.zeros((2, 3, Sq, (Skv + 3) // 4 * 4), device="cuda").bfloat16()
    padded[..., :Skv] = bias
    want = torch.empty_like(q)
    L = _lib.lib()
    qs, ks = _lib.strides_bhnd(Sq, 3, D), _lib.strides_bhnd(Skv, 3, D)
    ms = (ctypes.c_int64 * 4)(*padded.stride())
    assert L.mi355_sage_sdpa_bf16_mask(q.data_ptr(), k.data_ptr(), v.data_ptr(), padded.data_ptr(), want.data_ptr(), 2, 3, Sq, Skv, D, D ** -0.5,
                                       qs, ks, ks, ms, qs, 0, 0, 0, 0, 0, torch.cuda.current_stream().cuda_stream, variant, None, 0) == 0
    torch.cuda.synchronize()
    assert torch.isfinite(got.float()).all() and torch.equal(got, want)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16", "float16"])
def test_recorded_node_has_the_bits_of_the_python_node(dtype):
    """record_sdpa through the native node (F32, BF16; F16 falls through) against the Python node: values and gradients."""
    import torch
    from mojodiffusion_amd import attention_sage as A
    torch.manual_seed(1)
    base = [torch.randn((1, 130, 3, 64), device="cuda").to(getattr(torch, dtype)) for _ in range(4)]
    runs = []
    for fn in (A.record_sdpa, lambda q, k, v, s: A._SdpaNode.apply(q, k, v, s, A.PV_FP16)):
        q, k, v = (t.clone().requires_grad_(True) for t in base[:3])
        att = fn(q, k, v, 0.125)
        runs.append((att.detach(),) + torch.autograd.grad(att, (q, k, v), base[3].transpose(1, 2).contiguous().transpose(1, 2)))
    assert (_lib.host().record(*base[:3], 0.125, 0) is None) == (dtype == "float16")
    for a, b in zip(*runs):
        assert a.dtype == b.dtype and torch.equal(a, b)


def test_native_path_leaves_what_it_does_not_take():
    import torch
    from mojodiffusion_amd import attention_sage as A
    h = _lib.host()
    t = torch.zeros((1, 64, 2, 64), device="cuda").bfloat16()
    assert h.fwd(t, t, t, 0.1, 0, 0, 0, 0, 1) is not None
    for bad in (t.half(), t.cpu(), t.transpose(1, 2), t[0], None):
        assert h.fwd(bad, bad, bad, 0.1, 0, 0, 0, 0, 1) is None
    assert h.fwd(t, t, t, 0.1, 7, 0, 0, 0, 1) is None and h.fwd(t, t[:, :32].contiguous(), t[:, :32].contiguous(), 0.1, 0, 0, 0, 0, 1) is None
    with pytest.raises(A.Error, match="shim rc=-2"):
        A.sdpa_nomask(t, t, t, 0.1, 7)
    assert np.isfinite(A.sdpa_nomask(t.float(), t.float(), t.float(), 0.1).cpu().numpy()).all()


def test_subclasses_modes_and_exception_types():
    """A subclass's result is of its type, a mode sees plain tensors and leaves the shared workspace plain, running out of
    memory is torch's own exception: each as the Python path has it, with the native path's bits."""
    import torch
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.utils._python_dispatch import TorchDispatchMode
    from mojodiffusion_amd import attention_sage as A

    class Sub(torch.Tensor):
        pass

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    torch.manual_seed(2)
    t = torch.randn((1, 130, 2, 64), device="cuda").bfloat16()
    want = A.sdpa_nomask(t, t, t, 0.125)
    s = t.clone().as_subclass(Sub)
    got = A.sdpa_nomask(s, s, s, 0.125)
    assert type(got) is Sub and torch.equal(got.as_subclass(torch.Tensor), want)
    p = torch.nn.Parameter(t)
    assert type(A.sdpa_nomask(p, p, p, 0.125)) is torch.Tensor
    with Mode():
        assert _lib.host().fwd(t, t, t, 0.125, 0, 0, 0, 0, 1) is None
        assert torch.equal(A.sdpa_nomask(t, t, t, 0.125), want)
    with torch.cuda.stream(torch.cuda.Stream()):                # a stream without a workspace yet
        with FakeTensorMode() as fake:
            f = fake.from_tensor(t)
            with pytest.raises(RuntimeError):
                A.sdpa_nomask(f, f, f, 0.125)
        torch.cuda.synchronize()
        assert torch.equal(A.sdpa_nomask(t, t, t, 0.125), want)
    with pytest.raises(torch.OutOfMemoryError):
        _lib.host().workspace(1 << 50, t)
    torch.cuda.synchronize()
    assert torch.equal(A.sdpa_nomask(t, t, t, 0.125), want)


def test_threads_that_grow_workspaces_python_has_seen():
    """F16 storage takes the Python path, which sees the stream's workspace; the larger BF16 call behind it replaces that
    buffer natively.  Several threads at once, a stream each, finish with the results of one thread alone."""
    import threading
    import torch
    from mojodiffusion_amd import attention_sage as A
    torch.manual_seed(4)
    sizes = list(range(64, 1600, 96))
    x = [torch.randn((1, n, 2, 64), device="cuda") for n in sizes]
    call = lambda t: (A.sdpa_nomask(t.half(), t.half(), t.half(), 0.125), A.sdpa_nomask(t.bfloat16(), t.bfloat16(), t.bfloat16(), 0.125))
    want = [call(t) for t in x]
    torch.cuda.synchronize()
    got = {}

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            r = [call(t) for t in x]
            torch.cuda.current_stream().synchronize()
        got[i] = r

    threads = [threading.Thread(target=work, args=(i,), daemon=True) for i in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
        assert not t.is_alive(), "the threads wait for each other"
    for i in range(6):
        for a, b in zip(got[i], want):
            assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])


@pytest.mark.parametrize("entry", ["native", "python", "no_workspace"])
def test_threads_on_one_stream_share_its_workspace(entry):
    """Calls of several threads on one stream use one workspace: each has the bits of the call alone, forward, training
    forward and backward, through the native path, the Python path (F16 storage) and the library's own buffers."""
    import threading
    import torch
    from mojodiffusion_amd import attention_sage as A
    L = _lib.lib()
    torch.manual_seed(5)
    x = [[torch.randn((1, 700, 4, 64), device="cuda").bfloat16() for _ in range(2)] for _ in range(6)]
    qs = _lib.strides_bhnd(700, 4, 64)

    def call(t, g):
        if entry == "native":
            f = A.sdpa_flash_train_fwd(t, t, t, 0.125)
            b = A.sdpa_flash_backward(f, g, 0.125)
            return A.sdpa_nomask(t, t, t, 0.125), f.o, f.stats, b.d_q, b.d_k, b.d_v
        if entry == "python":
            return (A.sdpa_nomask(t.half(), t.half(), t.half(), 0.125),)
        o = torch.empty_like(t)
        assert L.mi355_sage_sdpa_bf16(t.data_ptr(), t.data_ptr(), t.data_ptr(), o.data_ptr(), 1, 4, 700, 700, 64, 0.125, qs, qs, qs, qs, 0, 0, 0, 0, 0,
                                      torch.cuda.current_stream().cuda_stream, 0, None, 0) == 0
        return (o,)

    want = [call(*p) for p in x]
    torch.cuda.synchronize()
    wrong = []

    def work(i):
        for rep in range(30):
            if not all(torch.equal(a, b) for a, b in zip(call(*x[i]), want[i])):
                wrong.append((i, rep))

    threads = [threading.Thread(target=work, args=(i,), daemon=True) for i in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
        assert not t.is_alive()
    assert not wrong, wrong


def test_recorded_node_under_saved_tensor_hooks():
    """The node saves through torch's hooks: a set that comes back as it was (from host memory, too) gives the same
    gradients; one that comes back as something else is refused before a kernel reads it."""
    import torch
    from mojodiffusion_amd import attention_sage as A
    torch.manual_seed(6)
    base = [torch.randn((1, 130, 3, 64), device="cuda").bfloat16() for _ in range(4)]

    def grads(pack, unpack):
        q, k, v = (t.clone().requires_grad_(True) for t in base[:3])
        with torch.autograd.graph.saved_tensors_hooks(pack, unpack):
            att = A.record_sdpa(q, k, v, 0.125)
        return torch.autograd.grad(att, (q, k, v), base[3])

    same = lambda t: t
    want = grads(same, same)
    for a, b in zip(grads(lambda t: t.cpu(), lambda t: t.cuda()), want):
        assert torch.equal(a, b)
    for unpack in (lambda t: t.cpu(), lambda t: t.half(), lambda t: t[:, :1], lambda t: t.transpose(1, 2), lambda t: t.float().contiguous()):
        with pytest.raises(RuntimeError):
            grads(same, unpack)

    class Mark(Exception):
        pass

    def fail(t):
        raise Mark("from the hook")
    with pytest.raises(Mark, match="from the hook"):
        grads(fail, same)
    for a, b in zip(grads(same, same), want):
        assert torch.equal(a, b)
