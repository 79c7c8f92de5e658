"""The fp32 matrix kernel behind every element type and size that the bf16 kernels do not take, at the edges of its tiles
(16 headdim rows or dstate columns per element of a lane's vector, at most 64), of its token groups (4 tokens a step, 64 a
window, a quarter of a chunk per wave) and on views that are only element-aligned, against the same sums in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    import ssd_amd
    from ssd_amd import _lib
    _lib.load()
    assert torch.cuda.is_available(), "these tests need the MI355X"
    return ssd_amd


def _chunk_states_64(d):
    """-> (chunk states, the sums of the absolute products) in 64 bits."""
    x, B, dt, dA, seq = d["x"].double(), d["B"].double(), d["dt"].double(), d["dA_cumsum"].double(), d["seq_idx"]
    b, L, H, P = x.shape
    G, N = B.shape[2:]
    C, Q = dt.shape[2:]
    B = B.repeat_interleave(H // G, dim=2)
    want, size = torch.zeros(b, C, H, P, N, dtype=torch.float64), torch.zeros(b, C, H, P, N, dtype=torch.float64)
    for c in range(C):
        t0, t1 = c * Q, min((c + 1) * Q, L)
        w = torch.exp(torch.clamp(dA[:, :, c, -1:] - dA[:, :, c, :t1 - t0], max=0.0)) * dt[:, :, c, :t1 - t0]
        if seq is not None:
            w = w * (seq[:, t0:t1] == seq[:, t1 - 1:t1])[:, None]
        xw = x[:, t0:t1].permute(0, 2, 3, 1) * w[:, :, None]
        Bc = B[:, t0:t1].permute(0, 2, 1, 3)
        want[:, c], size[:, c] = xw @ Bc, xw.abs() @ Bc.abs()
    return want, size


@pytest.mark.parametrize("kw", [
    dict(P=1, N=1, L=5, Q=4), dict(P=15, N=17, L=70, Q=64), dict(P=16, N=16, L=64, Q=64), dict(P=33, N=31, L=129, Q=128),
    dict(P=48, N=96, L=200, Q=100), dict(P=63, N=65, L=257, Q=256), dict(P=64, N=128, L=515, Q=256), dict(P=65, N=129, L=300, Q=300),
    dict(P=100, N=40, L=130, Q=65), dict(P=64, N=64, L=500, Q=64, b=6, H=32), dict(P=20, N=40, L=255, Q=64), dict(P=64, N=64, L=256, Q=64, b=5, H=77), dict(P=64, N=128, L=700, Q=128, b=8, H=64),
], ids=lambda kw: "-".join(f"{k}{v}" for k, v in kw.items()))
@pytest.mark.parametrize("dtype", ["fp32", "fp16", "bf16"])
def test_chunk_states_at_the_edges(ops, oracle, kw, dtype):
    args = dict(b=2, H=3, G=1, init=True, nseq=2 if kw["L"] > 128 else 0, dtype=dtype)
    args.update(kw)
    d = oracle.make_inputs(1, **args)
    print(f"[generic] {dtype} {kw}", flush=True)
    want, size = _chunk_states_64(d)
    # one element in front of every row: nothing but element alignment
    def shifted(t):
        wide = torch.zeros(*t.shape[:-1], t.shape[-1] + 1, dtype=t.dtype, device="cuda")
        wide[..., 1:] = t.cuda()
        return wide[..., 1:]
    x, B, dt, dA = shifted(d["x"]), shifted(d["B"]), d["dt"].cuda(), d["dA_cumsum"].cuda()
    seq = None if d["seq_idx"] is None else d["seq_idx"].cuda()
    b, C, H, P, N = want.shape
    buf = torch.full((b, C, H, P, N + 1), float("nan"), device="cuda")
    got = ops._chunk_state_fwd(B, x, dt, dA, seq_idx=seq, states=buf[..., 1:]).cpu()
    assert torch.isnan(buf[..., 0]).all()
    # every product and every addition rounds once (2^-24 of the sum of absolute products, Q additions at most), the
    # weight carries the rounding of its exponent (below 16) and of the exponential: 24 x 2^-24 covers both
    Q = d["dt"].shape[-1]
    assert ((got.double() - want).abs() <= (min(Q, args["L"]) + 32) * 2.0 ** -24 * size + 1e-30).all()
    # the fused call: chunk states + recurrence in place; 16-bit out: the walk over the chunks, or from four chunks on the
    # pair with a buffer of the wrapper's
    want_out, want_fin = oracle.fused_ref(d["B"], d["x"], d["dt"], d["dA_cumsum"], initial_states=d["initial_states"], seq_idx=d["seq_idx"])
    for out_dtype, rtol in ((torch.float32, 2e-3), (torch.float16, 2e-3), (torch.bfloat16, 1e-2)):
        out, fin = ops._fused_chunk_state_state_passing_fwd(B, x, dt, dA, out_dtype, initial_states=d["initial_states"].cuda(), seq_idx=seq)
        torch.testing.assert_close(out.float().cpu(), want_out.float(), rtol=rtol, atol=1e-3)
        torch.testing.assert_close(fin.cpu(), want_fin.float(), rtol=2e-3, atol=1e-3)


@pytest.mark.parametrize("Q", [64, 256])
def test_infinities_stay_where_they_are_and_tokens_behind_the_end_do_not_count(ops, oracle, Q):
    # an infinite x reaches its own headdim row only, and what lies behind a ragged end never enters a sum
    d = oracle.make_inputs(1, b=1, L=Q + 7, H=2, P=20, N=24, G=1, Q=Q, dtype="fp32", nseq=0, init=False)
    x = torch.full((1, 2 * Q, 2, 20), float("nan"))
    B = torch.full((1, 2 * Q, 1, 24), float("nan"))
    x[:, :Q + 7], B[:, :Q + 7] = d["x"], d["B"].abs() + 0.5
    x[0, Q + 2, 1, 3] = float("inf")
    d["x"], d["B"] = x[:, :Q + 7], B[:, :Q + 7]
    st = ops._chunk_state_fwd(B.cuda()[:, :Q + 7], x.cuda()[:, :Q + 7], d["dt"].cuda(), d["dA_cumsum"].cuda()).cpu()
    assert (st[0, 1, 1, 3] == float("inf")).all()
    st[0, 1, 1, 3] = 0.0
    want, _ = _chunk_states_64(d)
    want[0, 1, 1, 3] = 0.0
    torch.testing.assert_close(st.double(), want, rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("kw", [
    dict(P=80, N=128, L=2048, H=16, Q=128),                # tiles of 48 rows: row 77 ends one lane's vector and starts the next one's
    dict(P=80, N=128, L=2048, H=16, Q=128, dtype="bf16"), dict(P=63, N=65, L=257, Q=256), dict(P=31, N=24, L=300, Q=100, dtype="fp16"),
    dict(P=33, N=40, L=515, Q=128), dict(P=65, N=16, L=300, Q=300, dtype="bf16"), dict(P=77, N=129, L=700, Q=128),
    dict(P=63, N=128, L=700, Q=128, b=8, H=48),
], ids=lambda kw: "-".join(f"{k}{v}" for k, v in kw.items()))
def test_a_row_does_not_depend_on_where_it_lies(ops, oracle, kw):
    # Rows that two waves or workgroups hold (a lane's vector moved up to end at an odd headdim) are stored by both: the sums
    # must have one order.  All headdim rows of x hold the same numbers, so all rows of a state must hold the same bits.
    args = dict(b=1, H=3, G=1, init=False, nseq=0, dtype="fp32")
    args.update(kw)
    d = oracle.make_inputs(1, **args)
    print(f"[generic] same rows {kw}", flush=True)
    x, B, dt, dA = d["x"][..., :1].expand_as(d["x"]).contiguous().cuda(), d["B"].cuda(), d["dt"].cuda(), d["dA_cumsum"].cuda()
    same = lambda t: torch.equal(t, t[..., :1, :].expand_as(t))  # noqa: E731
    states = ops._chunk_state_fwd(B, x, dt, dA)
    assert float(states.abs().max()) > 0 and same(states)
    assert torch.equal(states, ops._chunk_state_fwd(B, x, dt, dA))
    calls = [ops._fused_chunk_state_state_passing_fwd(B, x, dt, dA, torch.float32)]
    old = ops.set_token_split(4)                           # the walk over the chunks
    try:
        calls += [ops._fused_chunk_state_state_passing_fwd(B, x, dt, dA, torch.float32) for _ in range(2)]
    finally:
        ops.set_token_split(old)
    for out, fin in calls:
        assert same(out) and same(fin)
    assert torch.equal(calls[1][0], calls[2][0]) and torch.equal(calls[1][1], calls[2][1])


def test_more_workgroups_than_one_launch_holds(ops):
    # chunks of one token: a tile per (token, head), four to a workgroup, 2^26 of them and some; one product each, rounded once
    L, H = (1 << 20) + 3, 64
    g = torch.Generator(device="cuda").manual_seed(5)
    x, B = torch.randn(1, L, H, 1, generator=g, device="cuda"), torch.randn(1, L, 1, 1, generator=g, device="cuda")
    dt, dA = torch.ones(1, H, L, 1, device="cuda"), torch.zeros(1, H, L, 1, device="cuda")
    print("[generic] 2^26 tiles", flush=True)
    assert torch.equal(ops._chunk_state_fwd(B, x, dt, dA)[..., 0], x * B)
