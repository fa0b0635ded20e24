"""The work that a user of the decay scan has it do, as measurable cases.

Three kinds of pass, each through the package's public functions:
  scan   the full-sequence scan of a prefill or an evaluation forward
         (``triton_global_decay`` / ``global_decay_scan``)
  train  the scan and its backward: y, dV and dlam
  step   one decode step for a batch (``decay_step``)

Inputs are synthetic: normal V (the projection's output under the model's
normalisation), decay factors drawn as the layer's sigmoid gives them, between
the half-life of one token (0.5) and of several thousand (0.9999; up to 0.99999
for long contexts).
"""
import math

import torch

import kilat_amd

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
SIZES = {"f32": 4, "bf16": 2, "f16": 2}

# Elements of V of the largest listed case (train_large); drawn cases stay below
# it by the work they do.
LARGEST = 16 * 16 * 4096 * 64


def _scan(name, B, H, N, D, dtype, **more):
    return dict({"name": name, "kind": "scan", "B": B, "H": H, "N": N, "D": D, "dtype": dtype, "out": dtype,
                 "layout": "heads", "final": False, "carry": False, "offset": 0, "lam_hi": 0.9999}, **more)


def _train(name, B, H, N, D, dtype, **more):
    return dict({"name": name, "kind": "train", "B": B, "H": H, "N": N, "D": D, "dtype": dtype,
                 "layout": "heads", "lam_hi": 0.9999}, **more)


def _step(name, B, H, D, dtype, per_sequence, in_place):
    return {"name": name, "kind": "step", "B": B, "H": H, "D": D, "dtype": dtype, "per_sequence": per_sequence,
            "in_place": in_place, "lam_hi": 0.9999}


def listed():
    return [
        # One user decoding: a single sequence's step in one layer of the
        # 12-head model (6 decay heads of 64 channels).  Launch and host cost.
        _step("step_one", 1, 6, 64, "bf16", per_sequence=False, in_place=False),
        # A serving pool's step: 256 sequences at positions of their own, the
        # state updated in place.
        _step("step_pool", 256, 12, 64, "bf16", per_sequence=True, in_place=True),
        # Prefill of one layer of that model: 8 sequences of 1024 tokens, V
        # as the projection leaves it, the decode state wanted too.
        _scan("prefill_layer", 8, 6, 1024, 64, "bf16", layout="tokens", final=True),
        # Short prompts filling the serving pool: 256 sequences of 200 tokens.
        _scan("prefill_prompts", 256, 12, 200, 64, "bf16", layout="tokens", final=True),
        # Chunked prefill: 1500 more tokens of 16 long sequences, from a
        # carried state at an offset, into fp32 outputs.
        _scan("prefill_chunk", 16, 12, 1500, 64, "bf16", out="f32", final=True, carry=True, offset=6000),
        # The headline workload: 8 sequences of 4096 tokens, 12 heads.
        _scan("scan_bf16", 8, 12, 4096, 64, "bf16"),
        # One long document: 65536 tokens, 16 heads of 128 channels.
        _scan("scan_long", 1, 16, 65536, 128, "bf16", lam_hi=0.99999),
        # Heads that are not a power of two: 1280 channels in 16 heads, fp16,
        # ragged length.
        _scan("scan_head80", 8, 16, 2047, 80, "f16", layout="tokens"),
        # A small fp32 training pass (fp32 parity configuration).
        _train("train_f32_small", 2, 6, 1024, 64, "f32"),
        # The headline workload as a training pass.
        _train("train_bf16", 8, 12, 4096, 64, "bf16"),
        # Training with 768 channels in 8 heads of 96, V and the gradient as
        # the projections lay them out, ragged length.
        _train("train_head96", 8, 8, 3001, 96, "bf16", layout="tokens"),
        # The larger sample configuration's decay heads (16 of 64 channels) at
        # a full training batch.
        _train("train_large", 16, 16, 4096, 64, "bf16"),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case: any batch, heads, length, head dim, dtype and layout."""
    kind = rng.choice(["scan", "scan", "scan", "train", "train", "step"])
    dtype = rng.choice(["bf16", "bf16", "f16", "f32"])
    H = rng.randint(1, 16)
    # Head dims of models in use: mostly multiples of 8, now and then one that
    # leaves rows off the 16-byte grid.
    D = rng.choice([16, 24, 32, 40, 48, 56, 64, 64, 64, 64, 72, 80, 96, 96, 100, 112, 128, 128, 160, 192, 256])
    lam_hi = rng.choice([0.999, 0.9999, 0.99999])
    if kind == "step":
        return {"kind": "step", "B": _log_int(rng, 1, 512), "H": H, "D": D, "dtype": dtype,
                "per_sequence": rng.random() < 0.5, "in_place": rng.random() < 0.5, "lam_hi": lam_hi}
    most = LARGEST // (2 if kind == "train" else 1) // (SIZES[dtype] // 2)
    N = _log_int(rng, 16, 65536)
    B = _log_int(rng, 1, max(1, min(256, most // (H * D * N))))
    N = max(16, min(N, most // (B * H * D)))
    case = {"kind": kind, "B": B, "H": H, "N": N, "D": D, "dtype": dtype,
            "layout": rng.choice(["heads", "tokens"]), "lam_hi": lam_hi}
    if kind == "scan":
        carry = rng.random() < 0.3
        case.update(out="f32" if rng.random() < 0.2 else dtype, final=rng.random() < 0.5, carry=carry,
                    offset=_log_int(rng, 1, 30000) if carry else 0)
    return case


def _lam(case, g):
    u = 0.5 + (case["lam_hi"] - 0.5) * torch.rand(case["H"], generator=g, device="cuda", dtype=torch.float64)
    # Heads that remember long are the common ones: push the draws towards 1.
    u = 1.0 - (1.0 - u) ** (1.0 + 2.0 * torch.rand(case["H"], generator=g, device="cuda", dtype=torch.float64))
    return u.clamp(max=case["lam_hi"]).float()


def _rows(case, g, dtype):
    """Normal [B, H, N, D] of `dtype`: contiguous ("heads"), or a view of the
    projection's [B, N, H*D] ("tokens")."""
    B, H, N, D = case["B"], case["H"], case["N"], case["D"]
    if case["layout"] == "tokens":
        return torch.randn(B, N, H, D, generator=g, device="cuda", dtype=dtype).permute(0, 2, 1, 3)
    return torch.randn(B, H, N, D, generator=g, device="cuda", dtype=dtype)


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    state = {"case": case, "lam": _lam(case, g)}
    dtype = DTYPES[case["dtype"]]
    B, H, D = case["B"], case["H"], case["D"]
    if case["kind"] == "step":
        state["state"] = 4.0 * torch.randn(B, H, D, generator=g, device="cuda")
        state["v"] = torch.randn(B, 1, H * D, generator=g, device="cuda", dtype=dtype)
        pos = torch.randint(1, 2049, (B,), generator=g, device="cuda", dtype=torch.int32)
        state["t_pos"] = pos if case["per_sequence"] else int(pos[0])
        return state
    state["V"] = _rows(case, g, dtype)
    if case["kind"] == "train":
        state["gy"] = _rows(case, g, dtype)
        state["V"].requires_grad_()
        state["lam"].requires_grad_()
    elif case["carry"]:
        state["carry"] = 4.0 * torch.randn(B, H, D, generator=g, device="cuda")
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "step":
        return kilat_amd.decay_step(state["lam"], state["state"], state["v"], state["t_pos"],
                                    new_state=state["state"] if case["in_place"] else None)
    if case["kind"] == "train":
        y = kilat_amd.triton_global_decay(state["lam"], state["V"])
        dV, dlam = torch.autograd.grad(y, (state["V"], state["lam"]), state["gy"])
        return {"y": y, "dV": dV, "dlam": dlam}
    if case["final"] or case["carry"] or case["out"] != case["dtype"]:
        return kilat_amd.global_decay_scan(
            state["lam"], state["V"], initial_state=state.get("carry"), return_final_state=case["final"],
            t_offset=case["offset"], out_dtype=DTYPES[case["out"]])
    return kilat_amd.triton_global_decay(state["lam"], state["V"])


def work(case):
    """Bytes: each call's inputs read once and its outputs written once.  A
    training pass is two calls: V in, y out; V and gy in, dV out.  Flops: a
    multiply-add per element of a scan and the scaling by 1/z; the backward's
    second scan, the gradient and its two sums over the rows."""
    es = SIZES[case["dtype"]]
    n = case["B"] * case["H"] * case["D"]
    if case["kind"] == "step":
        return {"bytes": n * (4 + es + 4 + 4), "flops": 3 * n}
    rows = n * case["N"]
    if case["kind"] == "train":
        return {"bytes": 5 * rows * es, "flops": 13 * rows}
    states = n * 4 * (int(case["final"]) + int(case["carry"]))
    return {"bytes": rows * (es + SIZES[case["out"]]) + states, "flops": 3 * rows}


def tolerance(case):
    """About four times what summing in another order showed (the sequential
    kernel against the chunked one, 26 scans of these ranges): 6e-5 for bf16
    outputs (the share of values that then round the other way), 8e-6 for
    fp16, 8e-7 for fp32 and for the fp32 states.  fp32 gradients: 1.4e-6
    against 64 bits, and dlam is a sum of both signs that may cancel further."""
    if case["kind"] == "step" or (case["kind"] == "scan" and case["out"] == "f32"):
        return {"rel": 4e-6}
    return {"rel": {"bf16": 2.5e-4, "f16": 5e-5, "f32": 1e-5}[case["dtype"]]}


def _z(lam, n, offset):
    """z of rows offset .. offset + n - 1 for every head, [H, n] in 64 bits."""
    e = torch.arange(offset + 1, offset + n + 1, device=lam.device, dtype=torch.float64)
    return (1.0 - lam[:, None] ** e) / ((1.0 - lam[:, None]) + 1e-6)


def _states(lam, V, s):
    """s_t = lam s_(t-1) + V_t for every row, in 64 bits, time first."""
    x = V.double().permute(2, 0, 1, 3).contiguous()
    a = lam[None, :, None]
    for t in range(x.shape[0]):
        s = x[t].addcmul_(a, s)
    return x


def exact(case, seed):
    state = prepare(case, seed)
    lam = state["lam"].detach().double()
    if case["kind"] == "step":
        B, H, D = case["B"], case["H"], case["D"]
        ns = lam[None, :, None] * state["state"].double() + state["v"].double().reshape(B, H, D)
        t = torch.as_tensor(state["t_pos"], device="cuda").double().reshape(-1, 1)
        z = (1.0 - lam ** (t + 1.0)) / ((1.0 - lam) + 1e-6)
        return ns / z[:, :, None], ns
    V = state["V"].detach()
    B, H, N, D = V.shape
    s0 = state["carry"].double() if state.get("carry") is not None else torch.zeros(B, H, D, device="cuda").double()
    s = _states(lam, V, s0)
    offset = case.get("offset", 0)
    rz = (1.0 / _z(lam, N, offset)).t()  # [N, H]
    y = (s * rz[:, None, :, None]).permute(1, 2, 0, 3)
    if case["kind"] == "scan":
        return (y, s[-1].clone()) if case["final"] else y
    gy = state["gy"].double().permute(2, 0, 1, 3)
    e = torch.arange(1, N + 1, device="cuda", dtype=torch.float64)[:, None]
    num, den = 1.0 - lam ** e, (1.0 - lam) + 1e-6
    # d(1/z)/dlam with 1/z = den / num
    dz = (-num + den * e * lam ** (e - 1.0)) / (num * num)
    dlam = (gy * s * dz[:, None, :, None]).sum(dim=(0, 1, 3))
    g = (gy * rz[:, None, :, None]).contiguous()
    a = lam[None, :, None]
    for t in range(N - 2, -1, -1):
        g[t].addcmul_(a, g[t + 1])
    dlam = dlam + (g[1:] * s[:-1]).sum(dim=(0, 1, 3))
    return {"y": y, "dV": g.permute(1, 2, 0, 3), "dlam": dlam}
