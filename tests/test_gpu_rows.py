"""The row kernels (kdecay_scan_fwd_rows and its backward): head dims and alignments the
channel-group kernels refuse, against the oracle and the sequential kernel."""
from __future__ import annotations

import pytest
import torch

import kilat_amd
from kilat_amd import _lib
from kilat_amd.triton_ops import _row_vectors_ok, chunked_head_dim
from oracle import decay_oracle as O
from tests.decay_cases import lam_uniform, rel_err
from tests.test_gpu_grad import check, gpu_grads, oracle_grads, rel

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16, "f64": torch.float64}
CODES = {"f32": _lib.KDECAY_F32, "bf16": _lib.KDECAY_BF16, "f16": _lib.KDECAY_F16, "f64": _lib.KDECAY_F64}
# The fp32 values differ in their last bits (1e-5 of the stream's largest), and
# where that moves one across a rounding boundary the 2-byte outputs differ by
# one ulp: 2^-8 to 2^-7 of the value for bf16 (8 significant bits), 2^-11 to
# 2^-10 for fp16 (11).
TOL = {torch.float32: 1e-5, torch.bfloat16: 1e-5 + 2.0 ** -7, torch.float16: 1e-5 + 2.0 ** -10, torch.float64: 1e-5}


@pytest.mark.parametrize("dname", ["f32", "bf16", "f16", "f64"])
def test_row_split_agrees_with_the_library(kdecay_lib, dname):
    """The shim's rule for which head dims the row kernel takes is the
    library's: it sizes a workspace for exactly those (several chunks here)."""
    for D in range(1, 700):
        ok = kdecay_lib.kdecay_scan_rows_workspace_bytes(2, 3, 100000, D, CODES[dname]) > 0
        assert ok == _row_vectors_ok(D, DTYPES[dname]), D


def test_rows_rejects_bad_arguments(kdecay_lib):
    fake = 0x100000
    ok = (3 * 4096 * 50, 4096 * 50, 50, 1)

    def call(V=fake, D=50, vstr=ok, ws=fake, wsb=1 << 30, code=_lib.KDECAY_BF16, ocode=_lib.KDECAY_BF16):
        return kdecay_lib.kdecay_scan_fwd_rows(V, code, _lib.strides4(vstr), fake, ocode, _lib.strides4(ok), fake, None,
                                               None, 2, 3, 4096, D, 0, ws, wsb, None)

    assert call(V=None) == _lib.KDECAY_EINVAL
    assert call(V=fake + 1) == _lib.KDECAY_ELAYOUT  # not on an element boundary
    assert call(vstr=(3 * 4096 * 100, 4096 * 100, 100, 2)) == _lib.KDECAY_ELAYOUT
    assert call(D=7) == _lib.KDECAY_ESHAPE  # less than one 16-byte vector
    assert call(code=9) == _lib.KDECAY_EDTYPE
    assert call(ocode=_lib.KDECAY_F16) == _lib.KDECAY_EDTYPE
    assert call(ws=None, wsb=0) == _lib.KDECAY_EWORKSPACE
    assert call(wsb=64) == _lib.KDECAY_EWORKSPACE
    assert call(ws=fake + 8) == _lib.KDECAY_EWORKSPACE


def _check(lam, V, dev, out_dtype=None, init=None, offset=0, out=None):
    lam_d, V_d = lam.to(dev), V.to(dev)
    if V_d.stride() != V.stride():
        V_d = torch.empty_strided(V.shape, V.stride(), dtype=V.dtype, device=dev).copy_(V)
    kw = dict(initial_state=None if init is None else init.to(dev), t_offset=offset, return_final_state=True,
              out_dtype=out_dtype)
    y, fin = kilat_amd.global_decay_scan(lam_d, V_d, **kw)
    yseq, fseq = kilat_amd.global_decay_scan(lam_d, V_d, algorithm="sequential", **kw)
    assert y.shape == V.shape and y.stride() == yseq.stride()
    tol = TOL[y.dtype]
    assert rel_err(y, yseq) <= tol and rel_err(fin, fseq) <= 1e-5
    if V.numel() <= 1 << 20:
        ref, sref = O.scan(lam, V.float() if V.dtype == torch.float64 else V, init, offset,
                           out_dtype=torch.float32 if y.dtype == torch.float64 else y.dtype)
        assert rel_err(y, ref) <= tol and rel_err(fin, sref) <= 1e-5
    return y


@pytest.mark.gpu
@pytest.mark.parametrize("dname,D", [
    ("bf16", 8), ("bf16", 9), ("bf16", 15), ("f16", 24), ("bf16", 33), ("f16", 40), ("bf16", 48), ("bf16", 50),
    ("f16", 80), ("bf16", 96), ("bf16", 100), ("f16", 127),  # one stream per head, 1 to 16 lanes
    ("bf16", 129), ("bf16", 136), ("f16", 160), ("bf16", 264), ("bf16", 301),  # two and three streams, surplus lanes
    ("f32", 4), ("f32", 5), ("f32", 20), ("f32", 50), ("f32", 63), ("f32", 68), ("f32", 100),
    ("f64", 2), ("f64", 3), ("f64", 20), ("f64", 33), ("f64", 50),
])
def test_rows_head_dims(hip_device, kdecay_lib, dname, D):
    """Every number of lanes per row; sequences of one row, around the end of a
    chunk of 8 rows per lane, and of several chunks; both layouts."""
    dtype = DTYPES[dname]
    assert _row_vectors_ok(D, dtype) and not chunked_head_dim(D, dtype)
    g = torch.Generator().manual_seed(900 + D)
    lam = lam_uniform(3, 0.5, 0.9999, g)
    vw = 16 // torch.empty((), dtype=dtype).element_size()
    nv = -(-D // vw)
    lpr = -(-nv // -(-nv // 16))
    L = 4 * (64 // lpr) * 8
    for N in (1, L - 1, L, L + 1, 5 * L + 3):
        for tokens in (False, True):
            V = torch.randn(2, N, 3, D, generator=g).to(dtype).transpose(1, 2)
            V = V if tokens else V.contiguous()
            init = torch.randn(2, 3, D, generator=g) if tokens else None
            _check(lam, V, hip_device, init=init, offset=7 if tokens else 0)


@pytest.mark.gpu
@pytest.mark.parametrize("dname,out,B,H,N,D", [
    ("bf16", None, 24, 16, 1500, 96),    # 16 rows per lane, several rounds
    ("f16", None, 8, 16, 2047, 80),      # one round
    ("bf16", "f32", 16, 9, 2000, 72),    # fp32 outputs, two stores per row
    ("f32", None, 16, 16, 1024, 40),
    ("bf16", None, 40, 10, 700, 50),     # 400 streams: counted through sub-counts
    ("f16", None, 1, 2, 30000, 40),      # a long chain: the wide window
    ("bf16", None, 130, 16, 60, 48),     # many short sequences
])
def test_rows_grids(hip_device, kdecay_lib, dname, out, B, H, N, D):
    g = torch.Generator().manual_seed(950 + D)
    lam = lam_uniform(H, 0.5, 0.9999, g)
    V = torch.randn(B, H, N, D, generator=g).to(DTYPES[dname])
    y1 = _check(lam, V, hip_device, out_dtype=DTYPES[out] if out else None)
    y2 = _check(lam, V, hip_device, out_dtype=DTYPES[out] if out else None)
    assert torch.equal(y1, y2)  # the same bits on every run


@pytest.mark.gpu
def test_rows_misaligned_views_and_out(hip_device, kdecay_lib):
    """D=64 (a head dim of the channel-group kernels) on bases and row strides
    off the 16-byte grid, and with out given: misaligned, with a channel
    stride, and V itself (written in place)."""
    g = torch.Generator().manual_seed(77)
    lam = lam_uniform(4, 0.8, 0.999, g).to(hip_device)
    big = torch.randn(2, 4, 900, 67, generator=g).to(torch.bfloat16).to(hip_device)
    for V in (big[..., 1:65], big[..., 3:53], big[:, :, 1::2, 2:66]):
        ref = kilat_amd.global_decay_scan(lam, V, algorithm="sequential")
        y = kilat_amd.triton_global_decay(lam, V)
        assert rel_err(y, ref) <= TOL[torch.bfloat16]
        room = torch.zeros(*V.shape[:3], V.shape[3] + 3, dtype=V.dtype, device=hip_device)
        out = room[..., 1:-2]
        assert kilat_amd.global_decay_scan(lam, V, out=out) is out and torch.equal(out, y)
        assert not room[..., 0].any() and not room[..., -2:].any()  # nothing written beside the rows
        wide = torch.zeros(*V.shape[:3], 2 * V.shape[3], dtype=V.dtype, device=hip_device)
        kilat_amd.global_decay_scan(lam, V, out=wide[..., ::2])
        assert torch.equal(wide[..., ::2], y) and not wide[..., 1::2].any()
        W = V.clone()
        kilat_amd.global_decay_scan(lam, W, out=W)
        assert rel_err(W, ref) <= TOL[torch.bfloat16]


def test_outputs_that_meet_an_input(kdecay_lib):
    """Which out= the kernels may not write directly: any that shares a byte range
    with an input, but V itself."""
    from kilat_amd import _native

    def meets(out, V, lam=torch.empty(3), init=None):
        assert _native.as_they_lie(lam, V, init, out) != _native.meets(out, V, lam, init)
        return _native.meets(out, V, lam, init)

    buf = torch.empty(2, 3, 11, 40)
    V = buf[:, :, 1:]
    assert not meets(V, V) and not meets(buf[:, :, 1:], V)
    assert meets(buf[:, :, :-1], V)  # shifted by a row
    assert meets(V.transpose(2, 3), V) and meets(V.view(torch.int32), V)
    assert not meets(torch.empty(2, 3, 10, 40), V)
    assert not meets(buf[1:], buf[:1]) and not meets(buf[:1], buf[1:])  # side by side
    lam, init = buf[0, 1, 5, :3], buf[:, :, 0]
    assert not meets(torch.empty(2, 3, 10, 40), V, lam, init) and meets(V, V, lam) and meets(V, V, init=init)
    assert not meets(buf[:, :, :0], V)


@pytest.mark.gpu
@pytest.mark.parametrize("D,base", [(80, 0), (50, 0), (64, 1), (64, 0)])
def test_out_that_overlaps_an_input(hip_device, kdecay_lib, D, base):
    """out= shifted by a row against V, over the carried state, and over one head
    only (several rows in the same memory, refused off the channel groups)."""
    lam = lam_uniform(4, 0.8, 0.999, torch.Generator().manual_seed(81)).to(hip_device)
    big = torch.randn(2, 4, 901, D + base, device=hip_device).to(torch.bfloat16)
    keep = big.clone()
    V, room = big[:, :, 1:, base:], big[:, :, :-1, base:]
    ref = kilat_amd.triton_global_decay(lam, V.clone())
    assert kilat_amd.global_decay_scan(lam, V, out=room) is room and rel_err(room, ref) <= TOL[torch.bfloat16]
    big.copy_(keep)
    f = torch.randn(2, 4, 30, D, device=hip_device)
    init, W = f[:, :, 0], torch.randn(2, 4, 30, D, device=hip_device)
    ref = kilat_amd.global_decay_scan(lam, W, initial_state=init.clone())
    kilat_amd.global_decay_scan(lam, W, initial_state=init, out=f)
    assert rel_err(f, ref) <= TOL[torch.float32]
    if D != 64:
        with pytest.raises(RuntimeError):
            kilat_amd.global_decay_scan(lam, W, out=torch.empty(2, 1, 30, D, device=hip_device).expand(2, 4, 30, D))


@pytest.mark.gpu
def test_rows_under_capture(hip_device, kdecay_lib):
    """Captured after reserve_workspace and replayed between eager calls of
    other shapes on the same workspace, the same bits."""
    g = torch.Generator().manual_seed(78)
    lam = lam_uniform(3, 0.8, 0.999, g).to(hip_device)
    V = torch.randn(2, 3, 3000, 80, generator=g).to(torch.bfloat16).to(hip_device)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert kilat_amd.triton_ops.reserve_workspace(2, 3, 3000, 80, torch.bfloat16, backward=False) > 0
        ref = kilat_amd.triton_global_decay(lam, V)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            y = kilat_amd.triton_global_decay(lam, V)
        for _ in range(3):
            y.zero_()
            graph.replay()
            kilat_amd.triton_global_decay(lam, V[:, :, :1000, :64])
            side.synchronize()
            assert torch.equal(y, ref)


def test_reserved_bytes_cover_the_route_of_every_head_dim(kdecay_lib):
    """reserve_workspace's size: never less than the row kernels', the
    channel-group kernels' or, for rows of less than one vector, the padded
    route's, forward and training."""
    from kilat_amd.triton_ops import _padded_head_dim, _reserve_bytes

    lib, B, H, N = kdecay_lib, 2, 3, 4096
    for dname, dtype in DTYPES.items():
        tname = "f32" if dname == "f64" else dname  # float64 is trained through the fp32 kernels
        for D in (1, 2, 3, 4, 7, 8, 16, 17, 32, 40, 64, 80, 96, 128, 129, 136):
            for train, name in ((False, dname), (True, tname)):
                rows, group = _row_vectors_ok(D, DTYPES[name]), chunked_head_dim(D, DTYPES[name])
                need = []
                if rows and not group:
                    need += [lib.kdecay_scan_rows_workspace_bytes, lib.kdecay_scan_rows_bwd_workspace_bytes][:1 + train]
                else:
                    need += [lib.kdecay_scan_workspace_bytes, lib.kdecay_scan_bwd_workspace_bytes][:1 + train]
                Dk = D if rows or group else _padded_head_dim(D, DTYPES[name])
                for size in need:
                    n = size(B, H, N, Dk, CODES[name])
                    assert 0 < n <= _reserve_bytes(lib, B, H, N, D, dtype, train), (dname, D, train)


@pytest.mark.gpu
@pytest.mark.parametrize("dname,D", [("bf16", 4), ("f32", 3), ("f16", 80), ("bf16", 16)])
def test_capture_after_reserve(hip_device, kdecay_lib, dname, D):
    """On a stream that ran nothing before, reserve_workspace suffices to capture
    a scan and a training pass; replayed between eager calls of other shapes."""
    dtype = DTYPES[dname]
    lam = lam_uniform(3, 0.8, 0.999, torch.Generator().manual_seed(79)).to(hip_device).requires_grad_()
    V = torch.randn(2, 4000, 3, D, device=hip_device).to(dtype).transpose(1, 2)
    _captured(lam, V, lambda: kilat_amd.reserve_workspace(2, 3, 4000, D, dtype))


def _captured(lam, V, prepare):
    """A forward and a training pass captured on a new stream after prepare(),
    every replay against the sequential kernel and an uncaptured backward."""
    gy = torch.randn_like(V)
    V = V.detach().requires_grad_()
    tol = TOL[V.dtype]
    with torch.no_grad():
        ref = kilat_amd.global_decay_scan(lam, V, algorithm="sequential")
    dv0, dl0 = torch.autograd.grad(kilat_amd.triton_global_decay(lam, V), (V, lam), gy)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        prepare()
        side.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            with torch.no_grad():
                y = kilat_amd.triton_global_decay(lam, V)
            yt = kilat_amd.triton_global_decay(lam, V)
            dv, dl = torch.autograd.grad(yt, (V, lam), gy)
        for _ in range(3):
            for t in (y, yt, dv, dl):
                t.detach().zero_()
            graph.replay()
            side.synchronize()
            for t in (y, yt.detach()):
                assert rel_err(t, ref) <= tol
            assert rel_err(dv, dv0) <= tol and rel(dl, dl0) <= 1e-4
            with torch.no_grad():  # eager, on the same workspace
                small = kilat_amd.triton_global_decay(lam, V[:, :, :100])
            assert rel_err(small, ref[:, :, :100]) <= tol
        assert kilat_amd.workspace_error(V) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,N,D,kind", [(20, 10, 230, 80, "padded"), (40, 12, 2000, 16, "narrow"),
                                          (20, 10, 2000, 16, "narrow"), (100, 12, 700, 64, "misaligned")])
def test_capture_on_a_workspace_too_small_for_the_row_kernels(hip_device, kdecay_lib, B, H, N, D, kind):
    """Where the stream's workspace holds what the route before the row kernels
    needs (zero-padding, the channel-group kernels on a view or on a copy) but
    not what they need, a capture takes that route, forward and training."""
    from kilat_amd.triton_ops import _padded_head_dim, _stream_ptr, _train_sizes, _workspace

    lib, code = kdecay_lib, _lib.KDECAY_BF16
    Dk = D if kind != "padded" else _padded_head_dim(D, torch.bfloat16)
    least = lib.kdecay_scan_workspace_least_bytes(B, H, N, Dk, code)
    rows = lib.kdecay_scan_rows_workspace_bytes(B, H, N, D, code)
    train, rows_train = (_train_sizes(lib, B, H, N, d, code, r)[1] for d, r in ((Dk, False), (D, True)))
    assert least < rows or train < rows_train
    lam = lam_uniform(H, 0.8, 0.999, torch.Generator().manual_seed(80)).to(hip_device).requires_grad_()
    V = torch.randn(B, N, H, D + (kind == "misaligned"), device=hip_device).to(torch.bfloat16).transpose(1, 2)
    V = V[..., 1:] if kind == "misaligned" else V
    if kind == "misaligned":  # trained through a copy in any case: the forward alone
        with torch.no_grad():
            ref = kilat_amd.global_decay_scan(lam, V, algorithm="sequential")
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                _workspace(hip_device, _stream_ptr(hip_device), least)
                side.synchronize()
                graph = torch.cuda.CUDAGraph()
                with torch.cuda.graph(graph, stream=side):
                    y = kilat_amd.triton_global_decay(lam, V)
                for _ in range(3):
                    y.zero_()
                    graph.replay()
                    side.synchronize()
                    assert rel_err(y, ref) <= TOL[torch.bfloat16]
        return
    _captured(lam, V, lambda: _workspace(hip_device, _stream_ptr(hip_device), max(least, train)))


def test_rows_backward_rejects_bad_arguments(kdecay_lib):
    fake = 0x100000
    ok = (3 * 4096 * 50, 4096 * 50, 50, 1)

    def call(V=fake, D=50, vstr=ok, states=fake, ws=fake, wsb=1 << 30, code=_lib.KDECAY_BF16):
        return kdecay_lib.kdecay_scan_rows_bwd(V, code, _lib.strides4(vstr), fake, _lib.strides4(ok), fake,
                                               _lib.strides4(ok), fake, None, states, None, fake, None, 2, 3, 4096, D,
                                               0, ws, wsb, None)

    assert call(V=None) == _lib.KDECAY_EINVAL
    assert call(V=fake + 1) == _lib.KDECAY_ELAYOUT
    assert call(vstr=(3 * 4096 * 100, 4096 * 100, 100, 2)) == _lib.KDECAY_ELAYOUT
    assert call(D=7) == _lib.KDECAY_ESHAPE
    assert call(code=_lib.KDECAY_F64) == _lib.KDECAY_EDTYPE
    assert call(states=None) == _lib.KDECAY_EINVAL
    assert call(ws=None, wsb=0) == _lib.KDECAY_EWORKSPACE
    assert call(wsb=4096) == _lib.KDECAY_EWORKSPACE


@pytest.mark.gpu
@pytest.mark.parametrize("dname,D", [
    ("bf16", 8), ("bf16", 9), ("f16", 24), ("bf16", 33), ("f16", 50), ("bf16", 80), ("bf16", 96), ("f16", 127),
    ("bf16", 136), ("f16", 160), ("bf16", 301), ("f32", 4), ("f32", 5), ("f32", 50), ("f32", 68), ("f32", 100),
])
def test_rows_backward_head_dims(hip_device, kdecay_lib, dname, D):
    """Every kind of row split (whole and shared last vectors, surplus lanes,
    one to three streams), sequences of one row, around the end of a chunk of
    4 rows per lane and of several chunks, with a carried state, a final-state
    gradient and an offset: against fp64 autograd through the oracle."""
    dtype = DTYPES[dname]
    g = torch.Generator().manual_seed(1000 + D)
    lam = lam_uniform(3, 0.5, 0.999, g)
    nv = -(-D // (16 // torch.empty((), dtype=dtype).element_size()))
    L = 4 * (64 // -(-nv // -(-nv // 16))) * 4
    for N, more in ((1, True), (L - 1, False), (L, True), (L + 1, False), (3 * L + 5, True)):
        V = torch.randn(2, 3, N, D, generator=g).to(dtype)
        gy = torch.randn(2, 3, N, D, generator=g).to(dtype)
        init = torch.randn(2, 3, D, generator=g) if more else None
        gfin = torch.randn(2, 3, D, generator=g) if more else None
        off = 9 if more else 0
        dv, dl, di = gpu_grads(lam, V, gy, hip_device, init=init, gfin=gfin, t_offset=off)
        rdv, rdl, rdi = oracle_grads(lam, V, gy, init=init, gfin=gfin, t_offset=off)
        check(dv, dl, di, rdv, rdl, rdi, dtype, f"D={D} N={N}")


@pytest.mark.gpu
@pytest.mark.parametrize("dname,B,H,N,D", [
    ("bf16", 4, 8, 1001, 96),    # 8 rows per lane, one round
    ("bf16", 9, 8, 2400, 96),    # 576 chunks of 16 rows per lane
    ("f16", 8, 9, 3300, 80),     # 648 of them, nine per stream: the wider window
    ("f32", 10, 12, 900, 50),    # 480 chunks at 16 rows: 8 rows, one round
    ("f16", 12, 10, 1500, 80),   # several rounds
    ("f32", 2, 3, 3000, 20),     # 4 rows per lane, chains of a few tens of chunks
    ("bf16", 1, 1, 9000, 100),   # a longer chain: the wide window
    ("bf16", 20, 12, 60, 48),    # 240 streams of one chunk
])
def test_rows_backward_grids(hip_device, kdecay_lib, dname, B, H, N, D):
    """From the projection layout, V and the gradient alike, against the
    channel-group kernels on zero-padded rows (padding changes no value; those
    kernels have their own tests against the oracle); the same bits on every
    run; gradients laid out like V."""
    dtype = DTYPES[dname]
    g = torch.Generator().manual_seed(1100 + D)
    lam = lam_uniform(H, 0.5, 0.999, g)
    V = torch.randn(B, N, H, D, generator=g).to(dtype).transpose(1, 2)
    gy = torch.randn(B, N, H, D, generator=g).to(dtype).transpose(1, 2)
    Dp = -(-D // 64) * 64
    V_p = torch.nn.functional.pad(V, (0, Dp - D)).to(hip_device).requires_grad_()
    lam_p = lam.to(hip_device).requires_grad_()
    y_p = kilat_amd.triton_global_decay(lam_p, V_p)
    rdv, rdl = torch.autograd.grad(y_p, (V_p, lam_p), torch.nn.functional.pad(gy, (0, Dp - D)).to(hip_device))
    rdv, rdl, y_p = rdv[..., :D].double().cpu(), rdl.cpu(), y_p.detach()[..., :D]
    first = None
    for _ in range(2):
        lam_d = lam.to(hip_device).requires_grad_()
        V_d = V.transpose(1, 2).to(hip_device).transpose(1, 2).requires_grad_()
        y = kilat_amd.triton_global_decay(lam_d, V_d)
        dv, dl = torch.autograd.grad(y, (V_d, lam_d), gy.transpose(1, 2).to(hip_device).transpose(1, 2))
        assert dv.stride() == V_d.stride() == y.stride()
        assert rel_err(y.detach(), y_p) <= TOL[dtype]
        check(dv.cpu(), dl.cpu(), None, rdv, rdl, None, dtype, f"grid D={D}")
        assert first is None or (torch.equal(first[0], dv) and torch.equal(first[1], dl))
        first = dv, dl


def _backward_chunks(lib, dname, B, H, N, D):
    """Chunks per stream of the row kernels' backward, from the size of its saved states."""
    n, rest = divmod(lib.kdecay_scan_rows_saved_states_floats(B, H, N, D, CODES[dname]) - 2 * H * N, B * H * D)
    assert rest == 0
    return n


def test_backward_rows_per_lane_fit_the_lds(kdecay_lib):
    """Grids of 513 to 768 chunks take 16 rows per lane, for which three
    workgroups have to fit a CU's LDS: rows of one lane (80 KB a workgroup) take 8."""
    for dname, D in (("bf16", 8), ("f16", 8), ("f32", 4)):
        assert _backward_chunks(kdecay_lib, dname, 10, 16, 16384, D) == 8  # 2048 rows: 8 per lane
    for dname, D in (("bf16", 16), ("f32", 8)):
        assert _backward_chunks(kdecay_lib, dname, 10, 16, 8192, D) == 4  # 2048 rows: 16 per lane


@pytest.mark.gpu
@pytest.mark.parametrize("dname,B,H,N,D", [("bf16", 40, 16, 4000, 8), ("f32", 40, 16, 4000, 4), ("bf16", 10, 16, 8000, 16)])
def test_rows_backward_of_one_and_two_lanes(hip_device, kdecay_lib, dname, B, H, N, D):
    """The grids of the test above: 8 rows per lane with one lane per row, 16 with two."""
    test_rows_backward_grids(hip_device, kdecay_lib, dname, B, H, N, D)


@pytest.mark.gpu
@pytest.mark.parametrize("dname,out,D", [("bf16", "f32", 96), ("bf16", None, 96), ("f16", "f32", 50), ("f64", None, 20),
                                         ("bf16", "f32", 3)])
def test_training_output_is_laid_out_like_V(hip_device, kdecay_lib, dname, out, D):
    """y of a training pass over a head dim off the channel groups has the
    strides of empty_like(V), also as fp32 of a 2-byte V and where V has a channel
    stride; the same values as from a contiguous V."""
    dtype, out = DTYPES[dname], DTYPES[out or dname]
    lam = lam_uniform(3, 0.5, 0.999, torch.Generator().manual_seed(4)).to(hip_device)
    wide = torch.randn(2, 130, 3, 2 * D, device=hip_device).to(dtype)
    for V in (wide[..., :D].contiguous().transpose(1, 2), wide.transpose(1, 2)[..., ::2],
              wide[..., :D].permute(0, 2, 3, 1).contiguous().transpose(2, 3)):
        W, C = V.detach().requires_grad_(), V.detach().contiguous().requires_grad_()
        y, ref = (kilat_amd.global_decay_scan(lam, v, out_dtype=out) for v in (W, C))
        assert y.dtype == out and torch.equal(y, ref)
        assert y.stride() == torch.empty_like(V, dtype=out).stride()
        gy = torch.randn_like(ref)
        assert torch.equal(torch.autograd.grad(y, W, gy)[0], torch.autograd.grad(ref, C, gy)[0])


@pytest.mark.gpu
def test_rows_backward_infinite_gradient_stays_in_its_channel(hip_device, kdecay_lib):
    """An infinite gradient at the last row: every earlier row of that channel
    is infinite (never NaN from rows past the end), the others are finite, also
    where a row's last vector repeats the channel."""
    for D, c in ((48, 0), (50, 45)):
        lam = torch.full((2,), 0.99, device=hip_device, requires_grad=True)
        V = torch.randn(1, 2, 77, D, device=hip_device).to(torch.bfloat16).requires_grad_()
        gy = torch.randn(1, 2, 77, D, device=hip_device).to(torch.bfloat16)
        gy[:, :, -1, c] = float("inf")
        dv, = torch.autograd.grad(kilat_amd.triton_global_decay(lam, V), V, gy)
        assert torch.isposinf(dv[..., c]).all()
        assert torch.isfinite(dv[..., :c]).all() and torch.isfinite(dv[..., c + 1:]).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dname,D", [("bf16", 16), ("bf16", 32), ("f16", 32), ("f32", 16)])
def test_narrow_heads_on_the_row_kernels(hip_device, kdecay_lib, dname, D):
    """Heads of 16 and 32 channels from the projection layout, large enough for
    the row kernels, against the chunked kernels that smaller batches of the same
    rows take: forward with a carried state, and the gradients."""
    from kilat_amd import _native

    dtype = DTYPES[dname]
    B, H, N = 6, 12, 2100
    B *= 64 // (D * torch.empty((), dtype=dtype).element_size())
    lam = lam_uniform(H, 0.5, 0.999, torch.Generator().manual_seed(9)).to(hip_device).requires_grad_()
    V = torch.randn(B, N, H, D, device=hip_device).to(dtype).transpose(1, 2)
    gy = torch.randn(B, N, H, D, device=hip_device).to(dtype).transpose(1, 2)
    init = torch.randn(B, H, D, device=hip_device)

    def call(rows):
        v = V[rows].requires_grad_()
        with torch.no_grad():
            y, fin = kilat_amd.global_decay_scan(lam, v, initial_state=init[rows], return_final_state=True, t_offset=3)
        dv, dl = torch.autograd.grad(kilat_amd.triton_global_decay(lam, v), (v, lam), gy[rows])
        return y, fin, dv, dl

    assert _native.narrow_rows(V) and not _native.narrow_rows(V[:1])
    y, fin, dv, dl = call(slice(None))
    parts = [call(slice(b, b + 1)) for b in range(B)]
    y0, fin0, dv0 = (torch.cat([p[k] for p in parts]) for k in range(3))
    dl0 = sum(p[3].double() for p in parts)
    assert rel_err(y, y0) <= TOL[dtype] and rel_err(fin, fin0) <= 1e-5 and rel_err(dv, dv0) <= TOL[dtype]
    assert float((dl - dl0).abs().max() / dl0.abs().max()) <= 1e-4


@pytest.mark.gpu
@pytest.mark.parametrize("dname,D,c", [("bf16", 48, 3), ("bf16", 50, 45), ("f32", 5, 2), ("bf16", 301, 295)])
def test_rows_backward_infinite_gradient_reaches_dlam(hip_device, kdecay_lib, dname, D, c):
    """An infinite gradient, of y or of the final state, leaves its head's dlam
    infinite or NaN (also in a channel that a row's last vector repeats, where
    it is NaN), the other head's finite and as without it."""
    lam = torch.tensor([0.5, 0.9], device=hip_device, requires_grad=True)
    V = torch.randn(1, 2, 402, D, device=hip_device).to(DTYPES[dname]).requires_grad_()
    gy = torch.randn(1, 2, 402, D, device=hip_device).to(DTYPES[dname])
    gfin = torch.randn(1, 2, D, device=hip_device)

    def dlam(gy, gfin):
        y, fin = kilat_amd.global_decay_scan(lam, V, return_final_state=True)
        return torch.autograd.grad((y, fin), lam, (gy, gfin))[0]

    ref = dlam(gy, gfin)
    assert torch.isfinite(ref).all()
    for where in ("y", "final"):
        g, f = gy.clone(), gfin.clone()
        (g[:, 0, 200] if where == "y" else f[:, 0])[..., c] = float("inf")
        dl = dlam(g, f)
        assert not torch.isfinite(dl[0]) and torch.equal(dl[1], ref[1])


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,N,D", [(1, 16, 32768, 80), (2, 8, 30000, 50), (40, 10, 3000, 96)])
def test_rows_give_up_is_flagged_not_hung(hip_device, kdecay_lib, B, H, N, D):
    """The row kernels' look-backs give up after one poll (the library's test
    hook): every launch returns and sets the error word, the one that gave up
    writes NaN where it has no carry, and every later one NaN everywhere until the
    workspace is cleared; then the first launch's bits.  16 streams, and 400, which
    count toward the epoch's advance through sub-counts."""
    lam = lam_uniform(H, 0.99, 0.9999, torch.Generator().manual_seed(44)).to(hip_device)
    V = torch.randn(B, N, H, D, device=hip_device).to(torch.bfloat16).transpose(1, 2)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())

    def call():
        y, fin = kilat_amd.global_decay_scan(lam, V, return_final_state=True)
        torch.cuda.synchronize()
        return y, fin, kilat_amd.workspace_error(V)

    with torch.cuda.stream(stream):
        ref, fref, err = call()
        assert err == 0 and bool(torch.isfinite(ref).all())
        kdecay_lib.kdecay_debug_set_spin_limit(1)
        gave_up = False
        try:
            for k in range(3):
                print(f"  forced give-up launch {k}", flush=True)
                y, fin, err = call()
                if gave_up:
                    assert bool(torch.isnan(y).all()) and bool(torch.isnan(fin).all()), k
                elif err:
                    assert bool(torch.isnan(y).any()), k
                    gave_up = True
                else:
                    assert torch.equal(y, ref), k
        finally:
            kdecay_lib.kdecay_debug_set_spin_limit(0)
        assert gave_up
        y, fin, err = call()
        assert bool(torch.isnan(y).all()) and bool(torch.isnan(fin).all()) and err == 1
        assert kilat_amd.workspace_error(V, clear=True) == 1
        for _ in range(2):  # the epoch advances again
            y, fin, err = call()
            assert err == 0 and torch.equal(y, ref) and torch.equal(fin, fref)


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,N,D", [(2, 4, 16384, 96), (16, 16, 1024, 80), (40, 10, 500, 50)])
def test_rows_backward_give_up_is_flagged_not_hung(hip_device, kdecay_lib, B, H, N, D):
    """The training pass likewise: its forward's and its reverse look-back and the
    wait for a head's dlam partials.  8 streams (the first chunk of each counts
    toward the epoch's advance), 256 and 400 (the head-summing workgroups and the
    last of each XCD do)."""
    g = torch.Generator().manual_seed(45)
    lam = lam_uniform(H, 0.9, 0.9999, g)
    V = torch.randn(B, H, N, D, generator=g).to(torch.bfloat16)
    gy = torch.randn(B, H, N, D, generator=g).to(torch.bfloat16)
    probe = V[:, :, :1].to(hip_device)  # selects the workspace of this device and stream
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())

    def call():
        dv, dl, _ = gpu_grads(lam, V, gy, hip_device)
        return dv, dl, kilat_amd.workspace_error(probe)

    with torch.cuda.stream(stream):
        dv0, dl0, err = call()
        assert err == 0
        kdecay_lib.kdecay_debug_set_spin_limit(1)
        gave_up = False
        try:
            for k in range(3):
                print(f"  forced give-up backward {k}", flush=True)
                dv, dl, err = call()
                if gave_up:
                    assert bool(torch.isnan(dv).all()) and bool(torch.isnan(dl).all()), k
                elif err:
                    assert bool(torch.isnan(dv).any()) or bool(torch.isnan(dl).any()), k
                    gave_up = True
        finally:
            kdecay_lib.kdecay_debug_set_spin_limit(0)
        assert gave_up
        dv, dl, err = call()
        assert bool(torch.isnan(dv).all()) and bool(torch.isnan(dl).all()) and err == 1
        assert kilat_amd.workspace_error(probe, clear=True) == 1
        for _ in range(2):
            dv, dl, err = call()
            assert err == 0 and torch.equal(dv, dv0) and torch.equal(dl, dl0)


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,N,D", [(2, 4, 3000, 80), (25, 10, 700, 96), (40, 10, 900, 50), (2, 3, 90, 80)])
def test_rows_training_pass_replays_from_a_graph(hip_device, kdecay_lib, B, H, N, D):
    """A training pass on the row kernels, captured and replayed with eager passes
    and scans on the same workspace between the replays: the eager bits every
    time (look-back words and dlam partials are tagged with the launch epoch).
    8, 250 and 400 streams of several chunks, and one chunk per stream."""
    g = torch.Generator().manual_seed(46)
    lam = lam_uniform(H, 0.5, 0.999, g).to(hip_device).requires_grad_()
    V = torch.randn(B, H, N, D, generator=g).to(torch.bfloat16).to(hip_device).requires_grad_()
    gy = torch.randn(B, H, N, D, generator=g).to(torch.bfloat16).to(hip_device)
    init = torch.randn(B, H, D, generator=g).to(hip_device).requires_grad_()

    def launch():
        y, fin = kilat_amd.global_decay_scan(lam, V, initial_state=init, return_final_state=True, t_offset=5)
        return (y, *torch.autograd.grad((y, fin), (V, lam, init), (gy, fin.detach())))

    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        ref = [t.detach().clone() for t in launch()]  # eager first: creates the workspace outside the capture
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            out = launch()
        torch.cuda.synchronize()
        for r in range(4):
            print(f"  training graph replay {r} N={N} D={D}", flush=True)
            for t in out:
                t.detach().zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert all(torch.equal(a.detach(), b) for a, b in zip(out, ref)), r
            again = launch()
            with torch.no_grad():
                kilat_amd.triton_global_decay(lam, V[:, :, : N // 2])
            torch.cuda.synchronize()
            assert all(torch.equal(a.detach(), b) for a, b in zip(again, ref)), r
        assert kilat_amd.workspace_error(V) == 0
