"""Chunks chosen by sequence length: one small chunk for short sequences, 384-row
chunks where 512-row ones would be three quarters full at most (and the edges of
both ranges), against the sequential kernel, forward and training."""
from __future__ import annotations

import pytest
import torch

import kilat_amd
from kilat_amd import _lib
from oracle import decay_oracle as O
from tests.decay_cases import lam_uniform, rel_err

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16, "f64": torch.float64}
# One ulp of the output type where the fp32 values (1e-5) round differently: at
# most 2^-7 of the value for bf16, 2^-10 for fp16.
TOL = {torch.float32: 1e-5, torch.bfloat16: 1e-5 + 2.0 ** -7, torch.float16: 1e-5 + 2.0 ** -10, torch.float64: 1e-5}


@pytest.mark.gpu
@pytest.mark.parametrize("dname,out,D,unit", [
    ("bf16", None, 64, 32), ("bf16", "f32", 64, 32), ("f16", None, 128, 32), ("f32", None, 32, 32),
    ("f64", None, 16, 32), ("bf16", None, 32, 64), ("f32", None, 16, 64), ("f16", None, 16, 128),
])
def test_short_sequences(hip_device, kdecay_lib, dname, out, D, unit):
    """unit: rows of the smallest chunk (4 rows x 1 wavefront).  Every chunk
    shape's last length and the next one's first, for few and for many streams,
    with a carried state, an offset and the final state; both layouts."""
    dtype = DTYPES[dname]
    g = torch.Generator().manual_seed(1200 + D)
    lengths = [1, 3, unit - 1, unit, unit + 1, 2 * unit, 2 * unit + 1, 4 * unit, 4 * unit + 1, 8 * unit, 8 * unit + 1,
               12 * unit, 12 * unit + 1, 16 * unit + 1, 24 * unit, 24 * unit + 1, 33 * unit, 36 * unit, 36 * unit + 1]
    for B, H in ((2, 3), (70, 7)):
        lam = lam_uniform(H, 0.5, 0.9999, g).to(hip_device)
        for N in lengths:
            V = torch.randn(B, N, H, D, generator=torch.Generator(device=hip_device).manual_seed(N), device=hip_device)
            V = V.to(dtype).transpose(1, 2)
            V = V if N % 2 else V.contiguous()
            init = torch.randn(B, H, D, device=hip_device)
            kw = dict(initial_state=init, t_offset=11, return_final_state=True, out_dtype=DTYPES[out] if out else None)
            y, fin = kilat_amd.global_decay_scan(lam, V, **kw)
            ys, fs = kilat_amd.global_decay_scan(lam, V, algorithm="sequential", **kw)
            assert rel_err(y, ys) <= TOL[y.dtype], (B, N)
            assert rel_err(fin, fs) <= 1e-5, (B, N)
    V = torch.randn(2, 3, 2 * unit + 5, D, generator=g).to(dtype)  # and once against the oracle
    lam = lam_uniform(3, 0.5, 0.9999, g)
    y = kilat_amd.triton_global_decay(lam.to(hip_device), V.to(hip_device))
    ref, _ = O.scan(lam, V.float() if dtype == torch.float64 else V)
    assert rel_err(y, ref) <= TOL[y.dtype]


def test_384_row_chunks_where_batch_slices_would_run(kdecay_lib):
    """384-row chunks in one launch take more words than the slices of 512-row
    chunks they replace: up to 72% of two chunks and three quarters of three."""
    lib = kdecay_lib
    for B, N, fit in ((100, 700, True), (64, 1025, True), (64, 1152, True), (64, 1153, False), (64, 513, True),
                      (64, 737, True), (64, 738, False)):
        sizes = [f(B, 12, N, 64, _lib.KDECAY_BF16)
                 for f in (lib.kdecay_scan_workspace_bytes, lib.kdecay_scan_workspace_least_bytes)]
        assert (sizes[0] > sizes[1]) == fit, (B, N)


@pytest.mark.gpu
@pytest.mark.parametrize("dname,out,H,D,N,streams", [
    ("bf16", None, 1, 64, 300, (160, 161, 512, 513)),             # one chunk per stream: small, two to a CU, more
    ("f32", None, 1, 64, 264, (255, 256, 257, 769)),              # two groups per head; the shortest length
    ("bf16", "f32", 1, 64, 350, (500, 1030, 1600)),               # fp32 outputs, also in slices
    ("f16", None, 2, 64, 700, (320, 322, 516)),                   # two chunks: 640, 644, 1032
    ("bf16", None, 1, 128, 600, (162, 256, 258, 384, 386)),       # two groups: 648, 1024, 1032, 1536, 1544
    ("f64", None, 1, 16, 1100, (139, 171, 256, 257)),             # fp64: 417, 513, 768, 771
    ("f16", "f32", 1, 64, 1100, (170, 171, 214, 342, 512, 513)),  # three chunks: 510, 513, 642, slices from 1026
])
def test_384_row_chunk_edges(hip_device, kdecay_lib, dname, out, H, D, N, streams):
    """Either side of the lines of 384-row chunks, against the sequential kernel."""
    for n in streams:
        lam = lam_uniform(H, 0.5, 0.9999, torch.Generator().manual_seed(n)).to(hip_device)
        V = torch.randn(n // H, H, N, D, device=hip_device).to(DTYPES[dname])
        kw = dict(return_final_state=True, out_dtype=DTYPES[out] if out else None)
        y, fin = kilat_amd.global_decay_scan(lam, V, **kw)
        ys, fs = kilat_amd.global_decay_scan(lam, V, algorithm="sequential", **kw)
        assert rel_err(y, ys) <= TOL[y.dtype] and rel_err(fin, fs) <= 1e-5, n


@pytest.mark.gpu
def test_small_workspace_takes_the_saving_shapes(hip_device, kdecay_lib):
    """A workspace of kdecay_scan_workspace_least_bytes, less than
    kdecay_scan_workspace_bytes for batches of 384-row chunks, still runs; one
    byte less is refused."""
    B, H, N, D = 100, 12, 700, 64
    lib = kdecay_lib
    least = lib.kdecay_scan_workspace_least_bytes(B, H, N, D, _lib.KDECAY_BF16)
    full = lib.kdecay_scan_workspace_bytes(B, H, N, D, _lib.KDECAY_BF16)
    assert 0 < least < full
    lam = lam_uniform(H, 0.5, 0.9999, torch.Generator().manual_seed(5)).to(hip_device)
    V = torch.randn(B, H, N, D, device=hip_device).to(torch.bfloat16)
    ref = kilat_amd.global_decay_scan(lam, V, algorithm="sequential")
    st = _lib.strides4(V.stride())
    stream = torch.cuda.current_stream().cuda_stream
    for nbytes, rc in ((full, 0), (least, 0), (least - 1, _lib.KDECAY_EWORKSPACE)):
        ws = torch.zeros(full, dtype=torch.uint8, device=hip_device)
        y = torch.zeros_like(V)
        assert lib.kdecay_scan_fwd(V.data_ptr(), _lib.KDECAY_BF16, st, y.data_ptr(), _lib.KDECAY_BF16, st,
                                   lam.data_ptr(), None, None, B, H, N, D, 0, ws.data_ptr(), nbytes, stream) == rc
        if rc == 0:
            assert rel_err(y, ref) <= TOL[torch.bfloat16]
            assert not ws[nbytes:].any()  # nothing past what was given


@pytest.mark.gpu
def test_capture_on_a_workspace_sized_for_longer_sequences(hip_device, kdecay_lib):
    """A workspace that sufficed for 512-row chunks in batch slices still does
    under capture, where it cannot grow."""
    lam = lam_uniform(12, 0.5, 0.9999, torch.Generator().manual_seed(6)).to(hip_device)
    V = torch.randn(100, 12, 700, 64, device=hip_device).to(torch.bfloat16)
    ref = kilat_amd.global_decay_scan(lam, V, algorithm="sequential")
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        kilat_amd.triton_ops.reserve_workspace(100, 12, 1000, 64, torch.bfloat16, backward=False)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            y = kilat_amd.triton_global_decay(lam, V)
        for _ in range(3):
            y.zero_()
            graph.replay()
            kilat_amd.triton_global_decay(lam, V[:, :, :600])
            side.synchronize()
            assert rel_err(y, ref) <= TOL[torch.bfloat16]


@pytest.mark.gpu
@pytest.mark.parametrize("dname,B,H,N,D", [
    ("bf16", 60, 7, 200, 64), ("f32", 40, 5, 300, 32), ("bf16", 100, 5, 33, 64), ("f16", 30, 12, 600, 64),
    ("bf16", 50, 6, 90, 128), ("bf16", 20, 4, 250, 16),
])
def test_training_of_short_sequences(hip_device, kdecay_lib, dname, B, H, N, D):
    """y, dV and dlam of short sequences against fp64 sums on the GPU."""
    dtype = DTYPES[dname]
    g = torch.Generator().manual_seed(1300 + N)
    lam = lam_uniform(H, 0.5, 0.999, g).to(hip_device).requires_grad_()
    V = torch.randn(B, N, H, D, device=hip_device).to(dtype).transpose(1, 2).requires_grad_()
    gy = torch.randn(B, N, H, D, device=hip_device).to(dtype).transpose(1, 2)
    y = kilat_amd.triton_global_decay(lam, V)
    dv, dl = torch.autograd.grad(y, (V, lam), gy)
    lam64, V64 = lam.detach().double().requires_grad_(), V.detach().double().requires_grad_()
    y64, _ = O.scan(lam64, V64)
    rdv, rdl = torch.autograd.grad(y64, (V64, lam64), gy.double())
    assert rel_err(y.detach(), y64.detach()) <= 2 * TOL[dtype]
    assert rel_err(dv, rdv) <= 2 * TOL[dtype]
    assert float((dl.double() - rdl).abs().max() / rdl.abs().max()) <= 1e-4
