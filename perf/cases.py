"""What this library is measured on: calls of its public entry points as a Mamba2 layer's program makes them.

A case is a dict of plain values:
  path    fused     _fused_chunk_state_state_passing_fwd_concurrent: chunk states + state passing (main.py's hot call)
          layer     dt preparation, the fused call, the state half of the chunk scan -- main.py's three calls in a row
          unfused   _chunk_state_fwd, then _state_passing_fwd
          scan      the fused call with the state half of the chunk scan, passed states not wanted
  b L H P N G Q     batch, tokens, heads, headdim, dstate, groups, chunk size
  dtype             of x, B, C (and of the raw dt): bf16, fp16 or fp32
  out               of the passed states: fp32, or a 16-bit type (the reference's out_dtype = C.dtype)
  init              initial states are given
  seqs              packed sequences per batch row (0: no seq_idx)
  decay             mamba: dt log-uniform in 1e-3 .. 1e-1, A in -16 .. -1;  slow: dt in 0.25 .. 1.25, A in -1 .. 0
"""
import math
import os
import sys

import torch

_PACKAGE = os.path.join(os.getcwd(), "mamba-fused-minimal_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(1, _PACKAGE)

import ssd_amd  # noqa: E402

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _case(name, path, b, L, H, P=64, N=128, G=1, Q=256, dtype="bf16", out="fp32", init=False, seqs=0, decay="mamba"):
    return dict(name=name, path=path, b=b, L=L, H=H, P=P, N=N, G=G, Q=Q, dtype=dtype, out=out, init=init, seqs=seqs, decay=decay)


def listed():
    return [
        # the smallest calls: the fp32 toy problem of the reference, and a short prompt through a small model's layer,
        # where launches and host work are most of the time
        _case("toy_fp32", "fused", 1, 1024, 8, N=64, dtype="fp32"),
        _case("short_prompt_layer", "layer", 1, 200, 24, out="bf16"),
        # the layer of the 130M model in training or batched prefill
        _case("layer_130m", "fused", 8, 2048, 24),
        # the layer of the 2.7B model: one row of the reference's own test case (all three calls, slow decay), a batch with
        # the states of a continued prefill, the two unfused calls, and the call whose passed states stay on chip
        _case("main_2p7b", "layer", 1, 2048, 80, out="bf16", decay="slow"),
        _case("layer_2p7b", "fused", 4, 8192, 80, init=True),
        _case("unfused_2p7b", "unfused", 4, 8192, 80, init=True),
        _case("scan_2p7b", "scan", 4, 8192, 80, init=True),
        # variable-length sequences packed into one row
        _case("packed_2p7b", "fused", 1, 32768, 80, seqs=16),
        # one very long sequence, grouped B
        _case("long_grouped", "fused", 1, 131072, 128, G=8),
        # half precision, a ragged last chunk; single precision; sizes off every tiling, grouped and packed
        _case("fp16_ragged", "fused", 2, 3001, 24, dtype="fp16", init=True),
        _case("fp32_130m", "fused", 2, 2048, 24, dtype="fp32"),
        _case("odd_sizes", "fused", 2, 1900, 15, P=48, N=96, G=3, Q=64, init=True, seqs=4),
    ]


def draw(rng):
    dtype = rng.choice(["bf16"] * 6 + ["fp16", "fp32"])
    path = rng.choice(["fused"] * 5 + ["layer"] * 2 + ["unfused", "scan"])
    G = rng.choice([1, 1, 1, 2, 8])
    H = G * max(1, round(math.exp(rng.uniform(math.log(4), math.log(128))) / G))
    P, N, Q = rng.choice([64, 64, 64, 128, 32]), rng.choice([128, 128, 64]), rng.choice([256, 256, 256, 128])
    if path == "fused" and rng.random() < 0.15:
        P, N, Q = rng.choice([16, 40, 48, 80, 96]), rng.choice([16, 24, 40, 96]), rng.choice([64, 100, 128])
    # the scan call without passed states is for bf16 and for groups of whole sets of four state tiles
    if path == "scan":
        dtype, H = "bf16", max(H, 4 * G) // (4 * G) * 4 * G
    tokens = math.exp(rng.uniform(math.log(128), math.log(131072)))
    # what a pass may cost: as much as the long grouped sequence on the matrix cores, a few milliseconds elsewhere
    most = 1.3e11 if dtype == "bf16" and P % 32 == 0 and N % 64 == 0 else 3e9
    tokens = min(tokens, most / (2 * H * P * N), 2.4e8 / (H * P))
    b = min(rng.choice([1, 1, 2, 3, 4, 8]), max(1, int(tokens) // 64))
    L = max(1, int(tokens) // b)
    if L >= Q and rng.random() < 0.5:
        L -= L % Q
    out = dtype if path == "layer" or (dtype == "bf16" and path == "fused" and rng.random() < 0.3) else "fp32"
    return dict(path=path, b=b, L=L, H=H, P=P, N=N, G=G, Q=Q, dtype=dtype, out=out, init=rng.random() < 0.4,
                seqs=rng.choice([0, 0, 2, 5]) if L >= 64 else 0, decay=rng.choice(["mamba", "mamba", "slow"]))


def prepare(case, seed):
    b, L, H, P, N, G, Q = (case[k] for k in "bLHPNGQ")
    dtype, dev = _DTYPES[case["dtype"]], torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)
    normal = lambda *size: torch.randn(size, generator=g, device=dev, dtype=dtype)  # noqa: E731
    uniform = lambda lo, hi, *size: torch.rand(size, generator=g, device=dev) * (hi - lo) + lo  # noqa: E731
    s = dict(case=case, x=normal(b, L, H, P), B=normal(b, L, G, N), out_dtype=_DTYPES[case["out"]], init=None, seq=None)
    if case["path"] in ("layer", "scan"):
        s["C"] = normal(b, L, G, N)
    # activated dt and A; the raw dt is what softplus and the bias turn into it
    if case["decay"] == "mamba":
        dt, A = torch.exp(uniform(math.log(1e-3), math.log(1e-1), b, L, H)), -torch.exp(uniform(0.0, math.log(16.0), H))
    else:
        dt, A = uniform(0.25, 1.25, b, L, H), -uniform(0.0, 1.0, H)
    s["A"] = A
    if case["path"] == "layer":
        s["bias"] = torch.full((H,), -4.6, device=dev)
        s["dt_raw"] = (dt + torch.log(-torch.expm1(-dt)) - s["bias"]).to(dtype)
    else:
        C = -(-L // Q)
        dt = torch.nn.functional.pad(dt, (0, 0, 0, C * Q - L)).view(b, C, Q, H).permute(0, 3, 1, 2).contiguous()
        s["dt"], s["dA"] = dt, torch.cumsum(dt * A.view(1, H, 1, 1), dim=-1)
    if case["init"]:
        s["init"] = 0.1 * torch.randn(b, H, P, N, generator=g, device=dev)
    if case["seqs"]:
        starts = torch.zeros(b, L, device=dev, dtype=torch.int32)
        starts.scatter_(1, torch.randint(1, L, (b, case["seqs"] - 1), generator=g, device=dev), 1)
        s["seq"] = torch.cumsum(starts, dim=1, dtype=torch.int32)
    return s


def run(s):
    c = s["case"]
    if c["path"] == "fused":
        return ssd_amd._fused_chunk_state_state_passing_fwd_concurrent(
            s["B"], s["x"], s["dt"], s["dA"], s["out_dtype"], initial_states=s["init"], seq_idx=s["seq"])
    if c["path"] == "layer":
        dA, dt = ssd_amd._chunk_cumsum_fwd(s["dt_raw"], s["A"], c["Q"], dt_bias=s["bias"], dt_softplus=True)
        out, final = ssd_amd._fused_chunk_state_state_passing_fwd_concurrent(
            s["B"], s["x"], dt, dA, s["out_dtype"], initial_states=s["init"], seq_idx=s["seq"])
        return dA, dt, out, final, ssd_amd._chunk_scan_states_fwd(s["C"], out, dA, seq_idx=s["seq"])
    if c["path"] == "unfused":
        states = ssd_amd._chunk_state_fwd(s["B"], s["x"], s["dt"], s["dA"], seq_idx=s["seq"])
        init = None if s["init"] is None else s["init"].flatten(-2)
        out, final = ssd_amd._state_passing_fwd(states.flatten(-2), s["dA"][..., -1], initial_states=init, seq_idx=s["seq"],
                                                chunk_size=c["Q"])
        return states, out, final
    _, final, y = ssd_amd._fused_chunk_state_state_passing_scan_fwd(
        s["B"], s["x"], s["C"], s["dt"], s["dA"], initial_states=s["init"], seq_idx=s["seq"], return_states=False)
    return final, y


def work(case):
    b, L, H, P, N, G, Q = (case[k] for k in "bLHPNGQ")
    C = -(-L // Q)
    size = lambda t: 4 if t == "fp32" else 2  # noqa: E731
    state, decay = b * H * P * N, b * H * C * Q * 4
    passed = state * C * size(case["out"])
    n = (b * L * H * P + b * L * G * N) * size(case["dtype"]) + state * 4          # x, B; final states
    n += (state * 4 if case["init"] else 0) + (b * L * 4 if case["seqs"] else 0)
    flops = 2 * b * L * H * P * N + 2 * C * state
    if case["path"] == "layer":       # each of the three calls reads its inputs and writes its outputs
        n += b * L * H * size(case["dtype"]) + 5 * decay + 2 * passed
    elif case["path"] == "unfused":
        n += 2 * decay + 3 * passed
    elif case["path"] == "scan":
        n += 2 * decay
    else:
        n += 2 * decay + passed
    if case["path"] in ("layer", "scan"):
        n += b * L * (G * N + H * P) * size(case["dtype"])                          # C; y
        flops += 2 * b * L * H * P * N
    return {"bytes": n, "flops": flops}


def tolerance(case):
    # 16-bit results: one rounding, at twice the error of the type at least; fp32 results: sums of 32-bit products, and with
    # bf16 operands x * w carried in 16 bits
    if "bf16" in (case["out"], case["dtype"] if case["path"] in ("layer", "scan") else ""):
        return {"rel": 7e-3}
    return {"rel": 1e-3 if case["out"] == "fp16" else 1e-5}


def exact(case, seed):
    """What run returns, computed chunk by chunk in 64 bits."""
    s = prepare(case, seed)
    b, L, H, P, N, G, Q = (case[k] for k in "bLHPNGQ")
    C, dev = -(-L // Q), s["x"].device
    A, seq = s["A"].double(), s["seq"]
    if case["path"] == "layer":
        raw = s["dt_raw"].double() + s["bias"].double()
        dt = torch.nn.functional.pad(torch.nn.functional.softplus(raw, threshold=1e9), (0, 0, 0, C * Q - L))
        dt = dt.view(b, C, Q, H).permute(0, 3, 1, 2).contiguous()
        dA = torch.cumsum(dt * A.view(1, H, 1, 1), dim=-1)
    else:
        dt, dA = s["dt"].double(), s["dA"].double()
    heads = lambda t: t.double().repeat_interleave(H // G, dim=2).transpose(1, 2).contiguous()  # noqa: E731  (b,k,G,N) -> (b,H,k,N)
    state = torch.zeros(b, H, P, N, device=dev, dtype=torch.float64) if s["init"] is None else s["init"].double()
    states = torch.empty(b, C, H, P, N, device=dev, dtype=torch.float64) if case["path"] == "unfused" else None
    out = torch.empty(b, C, H, P, N, device=dev, dtype=torch.float64) if case["path"] != "scan" else None
    y = torch.empty(b, L, H, P, device=dev, dtype=torch.float64) if "C" in s else None
    before = torch.zeros(b, device=dev, dtype=torch.int32)          # sequence of the token in front of the chunk
    for c in range(C):
        t0, t1 = c * Q, min((c + 1) * Q, L)
        ids = torch.zeros(b, t1 - t0, device=dev, dtype=torch.int32) if seq is None else seq[:, t0:t1]
        last = ids[:, -1]
        w = torch.exp(torch.clamp(dA[:, :, c, -1:] - dA[:, :, c, :t1 - t0], max=0.0)) * dt[:, :, c, :t1 - t0]
        w = w * (ids == last[:, None])[:, None]
        xw = (s["x"][:, t0:t1].double().permute(0, 2, 3, 1) * w[:, :, None]).contiguous()
        chunk = torch.matmul(xw, heads(s["B"][:, t0:t1]))
        if out is not None:
            out[:, c] = state
        if states is not None:
            states[:, c] = chunk
        if y is not None:
            scale = torch.exp(dA[:, :, c, :t1 - t0]) * (ids == before[:, None])[:, None]
            cy = torch.matmul(heads(s["C"][:, t0:t1]), state.transpose(-1, -2).contiguous())
            y[:, t0:t1] = (cy * scale[..., None]).transpose(1, 2)
        keep = torch.exp(dA[:, :, c, -1]) * (last == before)[:, None]
        state, before = keep[..., None, None] * state + chunk, last
    if case["path"] == "layer":
        return dA, dt, out, state, y
    if case["path"] == "unfused":
        return states, out.flatten(-2), state.flatten(-2)
    return (state, y) if case["path"] == "scan" else (out, state)
