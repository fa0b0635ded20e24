"""The host path in C++ (_native): it takes the calls whose arguments the kernels
read as they are, with the general path's results, and leaves the others to it."""
from __future__ import annotations

import os
import shutil
import subprocess
import sys

import pytest
import torch

import kilat_amd
from kilat_amd import triton_ops
from tests.decay_cases import lam_uniform

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16, "f64": torch.float64}


@pytest.mark.parametrize("dname", ["f32", "bf16", "f64"])
def test_head_dims_agree(kdecay_lib, dname):
    from kilat_amd import _native

    es = torch.empty((), dtype=DTYPES[dname]).element_size()
    for D in range(1, 700):
        assert _native.chunked_head_dim(D, es) == kilat_amd.chunked_head_dim(D, DTYPES[dname]), D


def test_cpu_and_foreign_arguments_are_left(kdecay_lib):
    from kilat_amd import _native

    lam, V = torch.rand(3), torch.randn(2, 3, 5, 64)
    assert _native.scan(lam, V, None, False, 0, None) is None
    assert _native.scan(lam, [1], None, False, 0, None) is None
    assert _native.scan(None, V, None, False, 0.0, None) is None
    assert _native.decay_step(lam, V[:, :, 0], V[:, :, 0], 3, None, None, torch.float32) is None
    with pytest.raises(RuntimeError, match="cpu"):
        kilat_amd.triton_global_decay(lam, V)


def test_narrow_heads_that_take_the_row_kernels(kdecay_lib):
    """Either side of the lines of narrow_rows, in the projection layout unless
    said; smaller than 4 MiB and rows of a whole memory line never."""
    from kilat_amd import _native

    def takes(B, H, N, D, dname="bf16", contiguous=False, **kw):
        V = torch.empty((B, H, N, D) if contiguous else (B, N, H, D), dtype=DTYPES[dname])
        return _native.narrow_rows(V if contiguous else V.transpose(1, 2), **kw)

    assert takes(8, 12, 1500, 32) and not takes(8, 12, 600, 32) and not takes(8, 12, 1500, 32, contiguous=True)
    assert not takes(8, 12, 1500, 64) and not takes(8, 12, 1500, 32, "f32") and takes(8, 12, 1500, 16, "f32")
    for N, fwd, train in ((3000, False, True), (8192, False, True), (8193, True, True), (32256, True, True)):
        assert takes(3, 13, N, 32) == fwd and takes(3, 13, N, 32, train=True) == train, N
    assert takes(5, 8, 2000, 32) and not takes(1, 12, 33000, 32) and takes(1, 13, 33000, 32)  # by streams, by rows in all
    assert takes(2, 10, 32768, 32, train=True) and not takes(2, 10, 32769, 32, train=True)
    assert takes(2, 12, 32769, 32, train=True)
    assert takes(2, 10, 16384, 16, "f32", train=True) and not takes(2, 10, 16385, 16, "f32", train=True)
    assert takes(2, 19, 28000, 16, "f32", train=True) and takes(4, 10, 16385, 16, "f32", train=True)
    for N, train in ((512, True), (513, False), (640, False), (641, True)):
        assert takes(20, 8, N, 32) and takes(20, 8, N, 32, train=True) == train, N
    assert takes(2, 12, 6000, 16) and not takes(1, 23, 6000, 16) and takes(1, 23, 12000, 16)
    assert takes(8, 12, 2000, 16, contiguous=True) and takes(8, 12, 2000, 16, wide=True)
    assert takes(16, 12, 1024, 16, contiguous=True, wide=True) and not takes(16, 12, 1025, 16, contiguous=True, wide=True)
    assert takes(8, 12, 2000, 16, contiguous=True, wide=True, train=True)


def test_package_imported_before_it_is_built(kdecay_lib, tmp_path):
    """Imported without its libraries the package raises at the first call, and
    works in the same process once they are there (build() and the fixtures that
    build import it first)."""
    src = os.path.dirname(kilat_amd.__file__)
    pkg = tmp_path / "kilat_amd"
    pkg.mkdir()
    for name in os.listdir(src):
        if name.endswith(".py"):
            shutil.copy(os.path.join(src, name), pkg)
    program = """
import shutil, sys
import torch, kilat_amd
assert kilat_amd.__file__.startswith(sys.argv[1]), kilat_amd.__file__
lam, V = torch.rand(3), torch.randn(2, 3, 5, 64)
calls = (lambda: kilat_amd.triton_global_decay(lam, V), lambda: kilat_amd.decay_step(lam, V[:, :, 0], V[:, :, 0], 3))
def error(call):
    try:
        call()
    except RuntimeError as e:
        return str(e)
for call in calls:
    assert "cannot be loaded" in error(call)
for name in ("libkdecay.so", "_native.so"):
    shutil.copy(sys.argv[2] + "/" + name, sys.argv[1] + "/kilat_amd/" + name)
for call in calls:
    assert "is on cpu" in error(call), error(call)
"""
    run = subprocess.run([sys.executable, "-c", program, str(tmp_path), src], capture_output=True, text=True,
                         env={**os.environ, "PYTHONPATH": str(tmp_path)}, cwd=tmp_path, timeout=300)
    assert run.returncode == 0, run.stderr


@pytest.mark.gpu
@pytest.mark.parametrize("dname,out,D", [("bf16", None, 64), ("bf16", "f32", 64), ("f16", None, 80), ("f32", None, 32),
                                         ("f32", None, 50), ("f64", None, 48), ("bf16", None, 16)])
def test_scan_equals_the_general_path(hip_device, kdecay_lib, dname, out, D):
    from kilat_amd import _native

    dtype, out = DTYPES[dname], DTYPES[out] if out else None
    g = torch.Generator().manual_seed(1400 + D)
    lam = lam_uniform(3, 0.5, 0.9999, g).to(hip_device)
    for N in (7, 700):
        for V in (torch.randn(2, 3, N, D, device=hip_device).to(dtype),
                  torch.randn(2, N, 3, D, device=hip_device).to(dtype).transpose(1, 2),
                  torch.randn(2, 3, 2 * N, D, device=hip_device).to(dtype)[:, :, ::2],
                  torch.randn(1, 3, N, D, device=hip_device).to(dtype).expand(2, 3, N, D)):
            for init in (None, torch.randn(2, 3, D, device=hip_device)):
                slow = triton_ops._scan(lam, V, init, True, 5, None, out, "chunked")  # also grows the workspace
                fast = _native.scan(lam, V, init, True, 5, out)
                assert fast is not None and all(torch.equal(a, b) for a, b in zip(fast, slow))
                assert fast[0].stride() == slow[0].stride() and fast[0].dtype == slow[0].dtype


@pytest.mark.gpu
def test_calls_left_to_the_general_path(hip_device, kdecay_lib):
    """Arguments that need a conversion, a copy, padding or an error."""
    from kilat_amd import _native

    lam = torch.rand(3, device=hip_device)
    V = torch.randn(2, 3, 40, 64, device=hip_device)
    init = torch.randn(2, 3, 64, device=hip_device)
    for args in ((lam.double(), V, None, False, 0, None), (lam[:2], V, None, False, 0, None),
                 (lam.cpu(), V, None, False, 0, None), (lam, V.int(), None, False, 0, None),
                 (lam, V[0], None, False, 0, None), (lam, V[:, :, :0], None, False, 0, None),
                 (lam, V[..., :3].contiguous(), None, False, 0, None), (lam, V[..., ::2], None, False, 0, None),
                 (lam, V, None, False, 2**64, None), (lam, V, init.half(), False, 0, None), (lam, V, init[..., :3], False, 0, None),
                 (lam, V, None, False, 0, torch.float16), (lam, V.double().requires_grad_(), None, False, 0, None)):
        assert _native.scan(*args) is None
    s, v = init, init.half()
    for args in ((lam, s.half(), v, 3, None, None, torch.float32), (lam, s, v.double(), 3, None, None, torch.float32),
                 (lam, s, v.transpose(0, 1), 3, None, None, torch.float32), (lam, s, v, 3.0, None, None, torch.float32),
                 (lam, s, v, 2**64, None, None, torch.float32),
                 (lam, s, v, torch.tensor([1, 2]), None, None, torch.float32),
                 (lam, s, v, 3, None, s[:1], torch.float32), (lam, s, v, 3, None, None, torch.float64)):
        assert _native.decay_step(*args) is None


@pytest.mark.gpu
def test_step_equals_the_general_path(hip_device, kdecay_lib):
    lam = lam_uniform(3, 0.5, 0.9999, torch.Generator().manual_seed(3)).to(hip_device)
    s = torch.randn(2, 3, 40, device=hip_device)
    pos = torch.tensor([4, 900], dtype=torch.int32, device=hip_device)
    for vt in (torch.float32, torch.bfloat16, torch.float16):
        v = torch.randn(2, 1, 120, device=hip_device).to(vt)
        for t_pos, same in ((9, torch.tensor([9, 9])), (pos, pos.cpu())):
            for ot in (torch.float32, torch.bfloat16):
                o, n = kilat_amd.decay_step(lam, s, v, t_pos, out_dtype=ot)
                o2, n2 = kilat_amd.decay_step(lam, s, v, same, out_dtype=ot)  # a host int64 vector: the general path
                assert torch.equal(o, o2) and torch.equal(n, n2) and o.dtype == ot
        out, state = torch.empty_like(o, dtype=torch.float32), s.clone()
        r = kilat_amd.decay_step(lam, state, v, pos, out=out, new_state=state)
        assert r[0] is out and r[1] is state and torch.equal(state, n)


@pytest.mark.gpu
def test_out_dtype_that_is_no_torch_dtype(hip_device, kdecay_lib):
    """What torch.empty_like takes for a dtype is taken (a Python type), and what
    it refuses is refused with its TypeError."""
    lam, V = torch.rand(3, device=hip_device), torch.randn(2, 3, 40, 16, dtype=torch.float64, device=hip_device)
    y = kilat_amd.global_decay_scan(lam, V, out_dtype=float)
    assert y.dtype == torch.float64 and torch.equal(y, kilat_amd.global_decay_scan(lam, V))
    for wrong in ("float64", 6, object()):
        with pytest.raises(TypeError):
            kilat_amd.global_decay_scan(lam, V, out_dtype=wrong)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 80, 16, 3])
def test_lazily_negated_views(hip_device, kdecay_lib, D):
    """Tensors whose memory holds their negation (torch._neg_view, the imaginary
    part of a conjugate) give what their values give: every input, out= and the
    upstream gradients."""
    lam = lam_uniform(3, 0.5, 0.9999, torch.Generator().manual_seed(D)).to(hip_device).requires_grad_()
    V, gy = (torch.randn(2, 3, 70, D, device=hip_device) for _ in range(2))
    init, gfin = (torch.randn(2, 3, D, device=hip_device) for _ in range(2))

    def neg(t):
        t = torch._neg_view(-t)
        assert t.is_neg()
        return t

    def call(view, algorithm="chunked"):
        v, i = view(V).requires_grad_(), view(init).requires_grad_()
        r = kilat_amd.global_decay_scan(lam, v, initial_state=i, return_final_state=True, algorithm=algorithm)
        return (*r, *torch.autograd.grad(r, (v, lam, i), (view(gy), view(gfin))))

    for algorithm in ("chunked", "sequential"):
        for a, b in zip(call(neg, algorithm), call(torch.clone, algorithm)):
            assert torch.equal(a, b)
        with torch.no_grad():
            ref = kilat_amd.global_decay_scan(lam, V, initial_state=init, algorithm=algorithm)
            out = neg(torch.zeros_like(V))
            y = kilat_amd.global_decay_scan(neg(lam), neg(V), initial_state=neg(init), out=out, algorithm=algorithm)
            assert y is out and torch.equal(out, ref)
    with torch.no_grad():
        assert torch.equal(kilat_amd.triton_global_decay(lam, neg(V)), kilat_amd.triton_global_decay(lam, V))
    for a, b in zip(kilat_amd.decay_step(neg(lam.detach()), neg(init), neg(gfin), 5),
                    kilat_amd.decay_step(lam.detach(), init, gfin, 5)):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 80, 3])
def test_training_pass_keeps_a_tensor_subclass(hip_device, kdecay_lib, D):
    """The result is of V's class, as without a gradient, and of a Parameter a
    plain tensor; the values and gradients are the plain tensor's."""
    class Sub(torch.Tensor):
        pass

    lam = torch.tensor([0.5, 0.9], device=hip_device, requires_grad=True)
    V, gy = torch.randn(2, 2, 50, D, device=hip_device, requires_grad=True), torch.randn(2, 2, 50, D, device=hip_device)
    y = kilat_amd.triton_global_decay(lam, V)
    z = kilat_amd.triton_global_decay(lam, V.as_subclass(Sub))
    assert type(z) is Sub and torch.equal(z.as_subclass(torch.Tensor), y)
    assert type(kilat_amd.triton_global_decay(lam.detach(), V.detach().as_subclass(Sub))) is Sub
    assert type(kilat_amd.triton_global_decay(lam, torch.nn.Parameter(V.detach()))) is torch.Tensor
    for a, b in zip(torch.autograd.grad(z, (V, lam), gy), torch.autograd.grad(y, (V, lam), gy)):
        assert torch.equal(a.as_subclass(torch.Tensor), b)


@pytest.mark.gpu
def test_training_pass_over_an_inference_tensor(hip_device, kdecay_lib):
    """V made under inference_mode: head dims off the channel groups take it (through
    a copy, which the backward can keep), those of the groups refuse it."""
    lam = torch.tensor([0.5, 0.9], device=hip_device, requires_grad=True)
    for D in (80, 64):
        V = torch.randn(2, 2, 50, D, device=hip_device)
        with torch.inference_mode():
            W = V.clone()
        if D == 64:
            with pytest.raises(RuntimeError, match="[Ii]nference"):
                kilat_amd.triton_global_decay(lam, W)
            continue
        y, z = kilat_amd.triton_global_decay(lam, V), kilat_amd.triton_global_decay(lam, W)
        assert torch.equal(y, z)
        assert torch.equal(torch.autograd.grad(z.sum(), lam)[0], torch.autograd.grad(y.sum(), lam)[0])


@pytest.mark.gpu
def test_gradients_of_an_empty_batch(hip_device, kdecay_lib):
    """No sequences, or no rows: dlam is zero."""
    for D in (64, 80, 3):
        for B, N in ((0, 5), (2, 0)):
            lam = torch.tensor([0.5, 0.9, 0.7], device=hip_device, requires_grad=True)
            V = torch.empty(B, 3, N, D, device=hip_device, requires_grad=True)
            y = kilat_amd.triton_global_decay(lam, V)
            junk = torch.full((3,), float("nan"), device=hip_device)
            del junk  # what an uninitialised dlam would be made of
            dl, dv = torch.autograd.grad(y, (lam, V), torch.empty_like(y))
            assert torch.equal(dl, torch.zeros_like(dl)) and dv.shape == V.shape


def _train_inputs(dev, D, seed=0):
    g = torch.Generator().manual_seed(seed)
    lam = lam_uniform(2, 0.5, 0.999, g).to(dev).requires_grad_()
    V, gy = (torch.randn(2, 2, 300, D, generator=g).to(dev) for _ in range(2))
    return lam, V.requires_grad_(), gy


def _grads(y, lam, V, gy):
    return torch.autograd.grad(y, (V, lam), gy)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 80])
def test_node_under_saved_tensor_hooks_and_checkpointing(hip_device, kdecay_lib, D):
    """Saved tensors that are packed elsewhere (copies, the host) or dropped and
    computed again give the same bits."""
    from torch.utils.checkpoint import checkpoint

    f = kilat_amd.triton_global_decay
    lam, V, gy = _train_inputs(hip_device, D)
    ref = _grads(f(lam, V), lam, V, gy)
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t) or t.clone(), lambda t: t):
        y = f(lam, V)
    assert any(t.data_ptr() == V.data_ptr() for t in packed)
    results = [_grads(y, lam, V, gy)]
    with torch.autograd.graph.save_on_cpu():
        y = f(lam, V)
    results += [_grads(y, lam, V, gy), _grads(checkpoint(f, lam, V, use_reentrant=False), lam, V, gy)]
    W = V.detach().clone().requires_grad_()
    checkpoint(f, lam, W, use_reentrant=True).backward(gy)
    results.append((W.grad, lam.grad))
    for dv, dl in results:
        assert torch.equal(dv, ref[0]) and torch.equal(dl, ref[1])


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 80])
def test_node_refusals(hip_device, kdecay_lib, D):
    """What the node cannot do raises: a second backward, V changed in place
    before the backward, functorch transforms, forward mode.  A backward with
    create_graph gives gradients without a graph."""
    import torch.autograd.forward_ad as fwad

    f = kilat_amd.triton_global_decay
    lam, V, gy = _train_inputs(hip_device, D)
    y = f(lam, V)
    _grads(y, lam, V, gy)
    with pytest.raises(RuntimeError, match="second time"):
        _grads(y, lam, V, gy)
    W = V * 1
    y = f(lam, W)
    W.add_(1)
    with pytest.raises(RuntimeError, match="inplace"):
        _grads(y, lam, V, gy)
    W, plain = V.detach(), lam.detach()
    for call in (lambda: torch.func.grad(lambda v: f(plain, v).sum())(W), lambda: torch.func.vjp(lambda v: f(plain, v), W),
                 lambda: torch.func.jvp(lambda v: f(plain, v), (W,), (gy,)),
                 lambda: torch.func.vmap(lambda v: f(plain, v))(torch.stack([W, W])),
                 lambda: torch.func.vmap(lambda v: kilat_amd.decay_step(plain, W[:, :, 0], v, 3)[0])(gy[:, :, :2].movedim(2, 0))):
        with pytest.raises(RuntimeError):
            call()
    with fwad.dual_level(), pytest.raises(RuntimeError):
        f(lam, fwad.make_dual(V, gy))
    dv, dl = torch.autograd.grad(f(lam, V), (V, lam), gy.clone().requires_grad_(), create_graph=True)
    assert not dv.requires_grad and not dl.requires_grad


@pytest.mark.gpu
def test_compiled_callers_break_the_graph_and_agree(hip_device, kdecay_lib):
    lam, V, gy = _train_inputs(hip_device, 64)
    step = (lam.detach(), V.detach()[:, :, 0].contiguous(), V.detach()[:, :, 1].contiguous(), 3)
    torch._dynamo.reset()
    for backend in ("eager", "aot_eager"):
        f = torch.compile(lambda a, v: 2 * kilat_amd.triton_global_decay(a, v * 1), backend=backend)
        y, ref = f(lam, V), 2 * kilat_amd.triton_global_decay(lam, V * 1)
        assert torch.equal(y, ref)
        for a, b in zip(_grads(y, lam, V, gy), _grads(ref, lam, V, gy)):
            assert torch.equal(a, b)
        g = torch.compile(lambda *a: kilat_amd.decay_step(*a)[0] + 1, backend=backend)
        assert torch.equal(g(*step), kilat_amd.decay_step(*step)[0] + 1)
    torch._dynamo.reset()


@pytest.mark.gpu
def test_threads_on_their_own_streams(hip_device, kdecay_lib):
    """Scans, training passes and steps from several threads at once, each on its
    own stream (and so its own workspace), give what one thread gives."""
    import threading

    data = [_train_inputs(hip_device, D, seed) for seed, D in enumerate((64, 80, 64, 50))]

    def work(lam, V, gy):
        y = kilat_amd.triton_global_decay(lam, V)
        with torch.no_grad():
            z, fin = kilat_amd.global_decay_scan(lam, V, return_final_state=True)
        s = kilat_amd.decay_step(lam.detach(), fin, gy[:, :, 0].contiguous(), 300)
        return (y.detach(), *_grads(y, lam, V, gy), z, fin, *s)

    ref = [work(*d) for d in data]
    torch.cuda.synchronize()
    errors = []

    def run(k):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(20):
                    out = work(*data[k])
                    torch.cuda.current_stream().synchronize()
                    assert all(torch.equal(a, b) for a, b in zip(out, ref[k]))
        except BaseException as e:  # noqa: B036 - reported by the main thread
            errors.append(e)

    threads = [threading.Thread(target=run, args=(k,)) for k in range(len(data))]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not errors and not any(t.is_alive() for t in threads), errors


@pytest.mark.gpu
def test_first_calls_of_two_threads(hip_device, kdecay_lib):
    """The first calls of a process, made by several threads at the same time,
    return (the workspace table is looked up once, which may let another thread run)."""
    program = """
import threading, torch, kilat_amd
lam, V = torch.rand(3, device="cuda"), torch.randn(2, 3, 3000, 64, device="cuda")
W, barrier, out = V.clone().requires_grad_(), threading.Barrier(6), []
def run(k):
    with torch.cuda.stream(torch.cuda.Stream()):
        barrier.wait()
        y = kilat_amd.triton_global_decay(lam, W if k % 2 else V)
        torch.cuda.current_stream().synchronize()
        out.append(y.detach())
torch.cuda.synchronize()
threads = [threading.Thread(target=run, args=(k,), daemon=True) for k in range(6)]
for t in threads: t.start()
for t in threads: t.join(60)
assert len(out) == 6
ref = kilat_amd.global_decay_scan(lam, V, algorithm="sequential")
assert all(((y - ref).abs().max() / ref.abs().max()).item() < 1e-5 for y in out)
"""
    root = os.path.dirname(os.path.dirname(kilat_amd.__file__))
    run = subprocess.run([sys.executable, "-c", program], cwd=root, capture_output=True, text=True, timeout=100)
    assert run.returncode == 0, run.stderr
