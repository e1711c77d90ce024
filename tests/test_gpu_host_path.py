"""The C++ host path of the inference calls (dkernel_amd/_host.so) against the Python launchers in
ops.py: same kernels, so every output bit must agree; and what it leaves to them (None) still works.
Also the tokens of packed inputs that belong to no sequence: their log-sum-exp reads -inf."""
import ctypes as C
import math

import pytest
import torch

from dkernel_amd import LocalStrideSparseAttention, SparseAttention, _lib, ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
New = LocalStrideSparseAttention.__wrapped__


class _PythonOnly:
    forward = paged = staticmethod(lambda *a: None)


def both(monkeypatch, call):
    """(result through _host, result through ops.py); asserts that _host took the call."""
    real, taken = _lib.host(), []

    class Spy:
        @staticmethod
        def forward(*a):
            taken.append(real.forward(*a))
            return taken[-1]

        @staticmethod
        def paged(*a):
            taken.append(real.paged(*a))
            return taken[-1]

    monkeypatch.setattr(_lib, "host", lambda: Spy)
    fast = call()
    assert len(taken) == 1 and taken[0] is not None, "the C++ path did not take this call"
    monkeypatch.setattr(_lib, "host", lambda: _PythonOnly)
    slow = call()
    monkeypatch.undo()
    return fast, slow


def same(a, b):
    a, b = (x if isinstance(x, tuple) else (x,) for x in (a, b))
    assert len(a) == len(b)
    for x, y in zip(a, b):
        assert x.shape == y.shape and x.dtype == y.dtype and x.stride() == y.stride() and torch.equal(x, y)


@pytest.mark.parametrize("dtype,D,bs,seq_dim,Hq,Hkv", [
    (torch.bfloat16, 128, 64, 1, 8, 2), (torch.float16, 64, 32, 2, 4, 4), (torch.float32, 64, 64, 1, 4, 2),
    (torch.bfloat16, 96, 128, 2, 6, 2), (torch.float32, 128, 32, 1, 2, 2)])
def test_unpadded_padded_and_single_token(monkeypatch, dtype, D, bs, seq_dim, Hq, Hkv):
    B, L = 3, 500
    print(f"case {dtype} D={D} bs={bs} seq_dim={seq_dim}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(1)
    mod = New(Hq, 512, bs, 2, 3, num_kv_heads=Hkv, seq_dim=seq_dim).to(DEV)

    def tensor(n, h):
        return torch.randn((B, n, h, D) if seq_dim == 1 else (B, h, n, D), generator=g, device=DEV).to(dtype)
    q, q1, k, v = tensor(L, Hq), tensor(1, Hq), tensor(L, Hkv), tensor(L, Hkv)
    lens = torch.tensor([500, 1, 333], dtype=torch.int32, device=DEV)
    for name, kw in (("plain", {}), ("left", dict(left_paddings=L - lens)), ("right", dict(seqlens=lens))):
        for x in (q, q1):
            for lse in (False, True):
                print(name, x.shape, lse, flush=True)
                same(*both(monkeypatch, lambda: mod(x, k, v, 0.1, return_lse=lse, **kw)))
    # left to the Python path: both lengths at once, lengths of another type, gradients
    for kw in (dict(left_paddings=L - lens, seqlens=lens), dict(seqlens=lens.long()), dict(left_paddings=(L - lens).cpu())):
        assert _lib.host().forward(q, k, v, 0.1, mod._buffers, mod._kernel_tables, mod.mask_lut_max_row, mod.kwargs, mod.seq_dim,
                                   None, None, kw.get("left_paddings"), kw.get("seqlens"), False, ops._impl, True) is None
        assert torch.isfinite(mod(q, k, v, 0.1, **kw).float()).all()
    out = mod(q.clone().requires_grad_(), k, v, 0.1)
    assert out.requires_grad


@pytest.mark.parametrize("Hq,Hkv,dtype,D", [(4, 2, torch.bfloat16, 128), (2, 2, torch.float32, 64), (3, 1, torch.float16, 40),
                                            (2, 2, torch.bfloat16, 20)])
def test_packed(monkeypatch, Hq, Hkv, dtype, D):
    print(f"case Hq={Hq} Hkv={Hkv} {dtype} D={D}", flush=True)
    lens, before, after = [70, 1, 200, 64], 5, 9
    T = before + sum(lens) + after
    g = torch.Generator(device=DEV).manual_seed(2)
    q, k, v = (torch.randn(T, h, D, generator=g, device=DEV).to(dtype) for h in (Hq, Hkv, Hkv))
    cu = torch.tensor([before] + [before + sum(lens[:i + 1]) for i in range(4)], dtype=torch.int32, device=DEV)
    mod = New(Hq, 256, 64, 2, 3, num_kv_heads=Hkv).to(DEV)
    fast, slow = both(monkeypatch, lambda: mod(q, k, v, 0.1, cu_seqlen_k=cu, return_lse=True))
    inside = slice(before, T - after)
    same((fast[0][inside], fast[1]), (slow[0][inside], slow[1]))
    assert torch.isinf(fast[1][:, :before]).all() and torch.isinf(fast[1][:, T - after:]).all()
    assert torch.isfinite(fast[1][:, inside]).all()
    # one query token per sequence (no offsets for the queries), and chunked prefill
    q1 = torch.randn(4, Hq, D, generator=g, device=DEV).to(dtype)
    same(*both(monkeypatch, lambda: mod(q1, k, v, 0.1, cu_seqlen_k=cu, return_lse=True)))
    cq = torch.tensor([0, 7, 8, 58, 60], dtype=torch.int32, device=DEV)
    qc = torch.randn(60, Hq, D, generator=g, device=DEV).to(dtype)
    same(*both(monkeypatch, lambda: mod(qc, k, v, 0.1, cu_seqlen_k=cu, cu_seqlen_q=cq, return_lse=True)))


def test_packed_tokens_without_any_sequence(monkeypatch):
    """Offsets of no sequence at all launch nothing; the log-sum-exps still read -inf, whatever the
    memory held before."""
    T, H, D = 300, 2, 64
    q, k, v = (torch.randn(T, H, D, device=DEV, dtype=torch.bfloat16) for _ in range(3))
    mod, cu = New(H, 512, 64, 2, 3).to(DEV), torch.zeros(1, dtype=torch.int32, device=DEV)
    empty = torch.empty

    def poisoned(*a, **kw):
        x = empty(*a, **kw)
        return x.fill_(float("nan")) if x.is_floating_point() else x
    monkeypatch.setattr(torch, "empty", poisoned)
    lse = mod(q, k, v, cu_seqlen_k=cu, return_lse=True)[1]
    assert lse.shape == (H, T) and torch.isneginf(lse).all()


@pytest.mark.parametrize("bs,fp8,dims", [(64, False, 3), (32, False, 4), (64, True, 3), (128, False, 3)])
def test_paged(monkeypatch, bs, fp8, dims):
    print(f"case bs={bs} fp8={fp8} dims={dims}", flush=True)
    B, Hq, Hkv, D, ps = 3, 8, 2, 128, 16
    g = torch.Generator(device=DEV).manual_seed(3)
    q = torch.randn(B, Hq, D, generator=g, device=DEV).to(torch.bfloat16)
    pools = [torch.randn(100, ps, Hkv, D, generator=g, device=DEV).to(torch.float8_e4m3fn if fp8 else torch.bfloat16) for _ in range(2)]
    table = torch.randperm(96, generator=g, device=DEV).to(torch.int32).view(3, 32)
    lens = torch.tensor([512, 1, 300], dtype=torch.int32, device=DEV)
    mod = New(Hq, 512, bs, 2, 3, num_kv_heads=Hkv).to(DEV)
    if dims == 4:
        q = q[:, None]
    for lse in (False, True):
        same(*both(monkeypatch, lambda: mod.paged_decode(q, *pools, table, lens, 0.1, return_lse=lse, k_scale=0.5)))


def test_launches_run_without_the_interpreter_lock():
    """PyGILState_Check in the place of dk_fwd, dk_fwd_paged and dk_bwd_balanced: its 0 for a thread that does not hold the
    lock reads as DK_OK, its 1 as a refusal, for which the C++ path returns None.  (Nothing is launched.)"""
    def address(f):
        return C.cast(f, C.c_void_p).value
    host, lib, check = _lib.host(), _lib.lib(), address(C.pythonapi.PyGILState_Check)
    mod = New(4, 256, 64, 2, 3, num_kv_heads=2).to(DEV)
    q, k, v = (torch.zeros(1, 256, h, 64, device=DEV, dtype=torch.bfloat16) for h in (4, 2, 2))
    n = torch.tensor([0, 256], dtype=torch.int32, device=DEV)
    tail = (mod._buffers, mod._kernel_tables, mod.mask_lut_max_row)
    csr = ops._lut((mod.layout_csr_crow, mod.layout_csr_col, 64, 64), q.device)
    csc = ops._lut((mod.layout_csc_ccol, mod.layout_csc_row, 64, 64), q.device)
    sizes = [address(lib.dk_fwd_workspace_bytes), address(lib.dk_bwd_balanced_workspace_bytes)]
    try:
        host.bind(check, sizes[0], check, check, sizes[1])
        res = [host.forward(q, k, v, 0.1, *tail, mod.kwargs, 1, None, None, None, None, True, ops._impl, True),
               host.forward(q[0], k[0], v[0], 0.1, *tail, mod.kwargs, 1, n, None, None, None, True, ops._impl, True),
               host.paged(q[:, 0], k.view(4, 64, 2, 64), v.view(4, 64, 2, 64), torch.arange(4, dtype=torch.int32, device=DEV)[None],
                          n[1:], 0.1, *tail, mod.lut_max_row, mod.lut_group, 256, True, 1.0, 1.0, ops._impl),
               host.train_forward(q, k, v, csr, 0.1, 1, True, ops._impl, True, True),
               host.train_backward(q, k, v, q, q, torch.zeros(1, 4, 256, device=DEV), None, None, None, None, csr, csc, ops._NO_LENGTHS, 0.1, 1,
                                   True, ops._impl, True)]
    finally:
        host.bind(address(lib.dk_fwd), sizes[0], address(lib.dk_fwd_paged), address(lib.dk_bwd_balanced), sizes[1])
    assert all(r is not None for r in res)


def test_user_pattern_and_errors():
    pat = torch.eye(4, dtype=torch.bool)
    mod = SparseAttention(64, pat).to(DEV)
    q, k, v = (torch.randn(1, 256, 2, 64, device=DEV, dtype=torch.bfloat16) for _ in range(3))
    assert mod(q, k, v).shape == q.shape
    with pytest.raises(AssertionError):
        mod(torch.cat([q, q], 1), torch.cat([k, k], 1), torch.cat([v, v], 1))  # longer than the pattern
    with pytest.raises(RuntimeError, match="ROCm"):
        mod(q.cpu(), k.cpu(), v.cpu())
    with pytest.raises(TypeError):
        mod(q.double(), k.double(), v.double())
    assert math.isfinite(mod(q[:, :0 + 1], k[:, :1], v[:, :1]).float().sum().item())


@pytest.mark.parametrize("dtype,D,bs,seq_dim,Hq,Hkv,fused,lse_grad", [
    (torch.bfloat16, 128, 64, 1, 8, 2, True, False), (torch.float16, 64, 32, 2, 4, 4, False, True),
    (torch.float32, 64, 64, 1, 4, 2, False, False), (torch.bfloat16, 96, 128, 2, 6, 2, False, True)])
def test_training_step(monkeypatch, dtype, D, bs, seq_dim, Hq, Hkv, fused, lse_grad):
    """Both halves of a training step through train_forward / train_backward and through ops.py: the same bits."""
    B, L = 2, 500
    print(f"case {dtype} D={D} bs={bs} seq_dim={seq_dim} fused={fused}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(1)
    mod = New(Hq, 512, bs, 2, 3, num_kv_heads=Hkv, seq_dim=seq_dim).to(DEV)

    def rand(h):
        return torch.randn((B, L, h, D) if seq_dim == 1 else (B, h, L, D), generator=g, device=DEV).to(dtype)

    if fused:
        xs = (rand(Hq + 2 * Hkv).requires_grad_(),)
    else:
        xs = tuple(rand(h).requires_grad_() for h in (Hq, Hkv, Hkv))
    dout, dlse = rand(Hq), torch.randn(B, Hq, L, generator=g, device=DEV)

    def step():
        if fused:
            out, lse = mod(xs[0], return_lse=True, split_qkv=lambda x: (x[:, :, :Hq], x[:, :, Hq:Hq + Hkv], x[:, :, Hq + Hkv:]))
        else:
            out, lse = mod(*xs, return_lse=True)
        return (out, lse) + torch.autograd.grad((out, lse) if lse_grad else out, xs, (dout, dlse) if lse_grad else dout)

    real, taken = _lib.host(), []

    class Spy:
        train_forward = staticmethod(lambda *a: taken.append(real.train_forward(*a)) or taken[-1])
        train_backward = staticmethod(lambda *a: taken.append(real.train_backward(*a)) or taken[-1])

    class Never:
        train_forward = train_backward = staticmethod(lambda *a: None)

    monkeypatch.setattr(_lib, "host", lambda: Spy)
    fast = step()
    assert len(taken) == 2 and all(x is not None for x in taken), "the C++ path did not take this step"
    monkeypatch.setattr(_lib, "host", lambda: Never)
    slow = step()
    monkeypatch.undo()
    same(tuple(x.detach() for x in fast), tuple(x.detach() for x in slow))


class _Subclass(torch.Tensor):
    pass


def test_training_step_left_to_ops(monkeypatch):
    """What the C++ halves refuse (None) and the launches of ops.py then do with the same bits: tensors of a subclass, a
    backward that is to be differentiated, a log-sum-exp gradient of another type; and gradient tensors of the caller's."""
    mod = New(2, 256, 64, 2, 3).to(DEV)
    xs = tuple(torch.randn(1, 256, 2, 64, device=DEV, dtype=torch.bfloat16, requires_grad=True) for _ in range(3))
    dout, dlse = torch.randn_like(xs[0]), torch.randn(1, 2, 256, device=DEV)
    real, taken = _lib.host(), []

    class Spy:
        train_forward = staticmethod(lambda *a: taken.append(real.train_forward(*a)) or taken[-1])
        train_backward = staticmethod(lambda *a: taken.append(real.train_backward(*a)) or taken[-1])

    def took(*what):  # of the calls since the last time: which ones the C++ halves did
        done, taken[:] = [x is not None for x in taken], []
        assert done == list(what), done

    monkeypatch.setattr(_lib, "host", lambda: Spy)
    out, lse = mod(*xs, return_lse=True)
    want = torch.autograd.grad((out, lse), xs, (dout, dlse), retain_graph=True)
    took(True, True)

    sub_out, sub_lse = mod(*(x.detach().as_subclass(_Subclass).requires_grad_() for x in xs), return_lse=True)
    took(False)
    assert torch.equal(sub_out, out) and torch.equal(sub_lse, lse)

    got = torch.autograd.grad((out, lse), xs, (dout, dlse), create_graph=True)
    took(False)
    same(got, want)
    assert not any(x.requires_grad for x in got)  # there is no second derivative to be had

    def backward(*a):
        with torch.no_grad():  # as autograd calls it
            return ops._backward(out.grad_fn, dout, *a)

    same(backward(dlse.double()), backward(dlse))
    took(False, True)

    # gradient tensors of the caller's: written in place where their rows are consecutive, refused otherwise
    given = [torch.zeros(1, 256, 2, 96, device=DEV, dtype=torch.bfloat16)[..., :64] for _ in range(3)]
    got = backward(dlse, *given)
    took(True)
    for a, b, w in zip(got, given, want):
        assert a.data_ptr() == b.data_ptr() and torch.equal(b, w)
    with pytest.raises(AssertionError):
        backward(dlse, torch.zeros(1, 256, 2, 128, device=DEV, dtype=torch.bfloat16)[..., ::2])
    took(False)

    # a gradient expanded from one value is laid out first, one of another type is cast by autograd: both ordinary steps
    a = torch.autograd.grad(out.sum(), xs, retain_graph=True)
    b = torch.autograd.grad(out, xs, torch.ones_like(out), retain_graph=True)
    same(a, b)
    same(torch.autograd.grad(lse.double().sum(), xs[:2], retain_graph=True), torch.autograd.grad(lse, xs[:2], torch.ones_like(lse)))
    took(True, True, True, True)
