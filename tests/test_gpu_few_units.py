"""Few state tiles and four or more chunks: chunk states + recurrence in front of the kernels that walk a sequence.  Both
sides of the rule's lines, every form of the call that it takes, against the token-split kernel on the same inputs and
against the oracle."""
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


@pytest.mark.parametrize("kw,pair", [
    (dict(L=1024, H=8), True),                             # four chunks
    (dict(L=768, H=8), False),                             # three
    (dict(L=1023, H=8, nseq=3), True),                     # ragged, packed
    (dict(L=2100, H=6, P=96, N=64), True),                 # a unit and a half of tiles, dstate 64
    (dict(L=1400, H=4, G=2, Q=128), True),                 # chunk 128, grouped B, ragged
    (dict(L=3840, H=51), True),                            # 25 units, 15 chunks: a tenth of 256, below three unit-chunks per compute unit
    (dict(L=2048, H=54), False),                           # 27 units
    (dict(L=16384, H=24), False),                          # three unit-chunks per compute unit, 12 units: the chain kernel
    (dict(L=24576, H=20), True),                           # ten units, any length
], ids=lambda v: "-".join(f"{k}{x}" for k, x in v.items()) if isinstance(v, dict) else str(v))
def test_few_units(ops, oracle, kw, pair):
    args = dict(b=1, P=64, N=128, G=1, Q=256, init=True, nseq=0)
    args.update(kw)
    d = oracle.make_inputs(1, **args)
    H, P, N, G, Q, L = (args[k] for k in "HPNGQL")
    assert (ops.fused_plan(1, L, H, P, N, G, Q, compute_units=256)["family"] == "pair") == pair
    mv = lambda t: None if t is None else t.cuda()  # noqa: E731
    x, B, dt, dA, seq, init = (mv(d[k]) for k in ("x", "B", "dt", "dA_cumsum", "seq_idx", "initial_states"))
    print(f"[few] {kw}", flush=True)
    fused = ops._fused_chunk_state_state_passing_fwd
    old = ops.set_token_split(4)
    try:
        want, want_fin = fused(B, x, dt, dA, torch.float32, initial_states=init, seq_idx=seq)
        want_y = ops._chunk_scan_states_fwd(mv(d["C"]), want, dA, seq_idx=seq, out_dtype=torch.float32)
    finally:
        ops.set_token_split(old)
    o_out, o_fin = oracle.fused_ref(d["B"], d["x"], d["dt"], d["dA_cumsum"], initial_states=d["initial_states"], seq_idx=d["seq_idx"])
    torch.testing.assert_close(want.cpu(), o_out, rtol=2e-3, atol=1e-3)
    torch.testing.assert_close(want_fin.cpu(), o_fin, rtol=2e-3, atol=1e-3)
    # both sides split x * w into bf16 hi + lo (2^-17 of every product) and add in fp32 in another order
    tol = dict(rtol=1e-4, atol=1e-4)
    for out_dtype in (torch.float32, torch.bfloat16, torch.float16):
        out, fin = fused(B, x, dt, dA, out_dtype, initial_states=init, seq_idx=seq)
        assert out.dtype == out_dtype and fin.dtype == torch.float32
        torch.testing.assert_close(fin.cpu(), o_fin, rtol=2e-3, atol=1e-3)
        if out_dtype == torch.float32:
            torch.testing.assert_close(out, want, **tol)
            torch.testing.assert_close(out.cpu(), o_out, rtol=2e-3, atol=1e-3)
        else:
            torch.testing.assert_close(out.float(), want, rtol=2.0 ** (-7 if out_dtype == torch.bfloat16 else -10), atol=1e-4)
        torch.testing.assert_close(fin, want_fin, **tol)
    # a states buffer of the caller, the scan's state half behind it, a captured call replayed between eager ones
    states = torch.full(want.shape, float("nan"), device="cuda")
    out, fin = fused(B, x, dt, dA, torch.float32, initial_states=init, seq_idx=seq, states=states)
    torch.testing.assert_close(out, want, **tol)
    torch.testing.assert_close(states, ops._chunk_state_fwd(B, x, dt, dA, seq_idx=seq), **tol)
    if H * P // 32 % 4 == 0 and H // G * P // 32 % 4 == 0:
        none, fin, y = ops._fused_chunk_state_state_passing_scan_fwd(B, x, mv(d["C"]), dt, dA, initial_states=init, seq_idx=seq,
                                                                     return_states=False, y_dtype=torch.float32)
        assert none is None
        torch.testing.assert_close(fin, want_fin, **tol)
        torch.testing.assert_close(y, want_y, rtol=1e-3, atol=1e-3)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        g_out, g_fin = fused(B, x, dt, dA, torch.bfloat16, initial_states=init, seq_idx=seq)
    for _ in range(3):
        g_out.zero_()
        g_fin.zero_()
        graph.replay()
        eager, eager_fin = fused(B, x, dt, dA, torch.bfloat16, initial_states=init, seq_idx=seq)
        torch.cuda.synchronize()
        assert torch.equal(g_out, eager) and torch.equal(g_fin, eager_fin)


def test_a_strided_initial_plane_keeps_the_kernel_it_had(ops, oracle):
    # initial states out of a wider cache: the recurrence walks a head's plane as one row and cannot take them, so no buffer
    # is made and the chain kernel serves bf16 `out` as it would without the rule (32 chunks of 8 heads)
    d = oracle.make_inputs(1, b=1, L=8192, H=8, init=True)
    x, B, dt, dA = (d[k].cuda() for k in ("x", "B", "dt", "dA_cumsum"))
    init = torch.zeros(1, 8, 64, 160, device="cuda")[..., :128]
    init.copy_(d["initial_states"])
    want_out, want_fin = oracle.fused_ref(d["B"], d["x"], d["dt"], d["dA_cumsum"], initial_states=d["initial_states"])
    ops.release_workspaces()
    out, fin = ops._fused_chunk_state_state_passing_fwd(B, x, dt, dA, torch.bfloat16, initial_states=init)
    torch.cuda.synchronize()
    from ssd_amd.ops import _WORKSPACES
    assert [k.epochs.last for k in _WORKSPACES.values()] == [1] and ops.fused_status() == 0
    torch.testing.assert_close(out.float().cpu(), want_out, rtol=2.0 ** -7, atol=1e-3)
    torch.testing.assert_close(fin.cpu(), want_fin, rtol=2e-3, atol=1e-3)
    # where only the fp32 matrix kernel applies: its walk, no buffer beside it
    y, yf = ops._fused_chunk_state_state_passing_fwd(B.half(), x.half(), dt, dA, torch.float16, initial_states=init)
    torch.testing.assert_close(y.float().cpu(), want_out, rtol=2e-3, atol=1e-3)
    torch.testing.assert_close(yf.cpu(), want_fin, rtol=2e-3, atol=1e-3)


# chain: of the calls with fp32, bf16 and no passed states, which run the chain kernel
@pytest.mark.parametrize("nseq,L,H,chain", [(7, 26624, 8, (1, 1, 1)), (0, 26624, 8, (0, 0, 0)), (7, 16384, 8, (0, 0, 0)), (5, 9216, 24, (0, 0, 1)),
                                            (5, 24576, 4, (0, 1, 0)), (5, 7936, 48, (0, 0, 1)), (5, 4352, 48, (0, 0, 0))])
def test_packed_rows_run_the_chain_kernel_beyond_the_packed_line(ops, oracle, nseq, L, H, chain):
    d = oracle.make_inputs(1, b=1, L=L, H=H, init=True, nseq=nseq)
    mv = lambda t: None if t is None else t.cuda()  # noqa: E731
    args = [mv(d[k]) for k in ("B", "x", "dt", "dA_cumsum")]
    kw = dict(initial_states=mv(d["initial_states"]), seq_idx=mv(d["seq_idx"]))
    want_out, want_fin = oracle.fused_ref(d["B"], d["x"], d["dt"], d["dA_cumsum"], initial_states=d["initial_states"], seq_idx=d["seq_idx"])
    from ssd_amd.ops import _WORKSPACES
    calls = [lambda o=o: ops._fused_chunk_state_state_passing_fwd(*args, o, **kw) for o in (torch.float32, torch.bfloat16)]
    calls.append(lambda: ops._fused_chunk_state_state_passing_scan_fwd(args[0], args[1], mv(d["C"]), *args[2:], return_states=False, **kw))
    for call, on_chain in zip(calls, chain):
        ops.release_workspaces()
        got = call()
        torch.cuda.synchronize()
        assert max((k.epochs.last for k in _WORKSPACES.values()), default=0) == on_chain and ops.fused_status() == 0
        torch.testing.assert_close(got[1].cpu(), want_fin, rtol=2e-3, atol=1e-3)
        if got[0] is not None:
            torch.testing.assert_close(got[0].float().cpu(), want_out, rtol=2e-3 if got[0].dtype == torch.float32 else 2.0 ** -7, atol=1e-3)


def test_without_room_for_chunk_states_the_call_runs_on_its_former_kernel(ops, oracle, monkeypatch):
    # 8 heads x 32 chunks: bf16 out and the scan call on the chain kernel, fp16 on the walk of the fp32 matrix kernel
    d = oracle.make_inputs(1, b=1, L=8192, H=8, init=True)
    x, B, C, dt, dA, init = (d[k].cuda() for k in ("x", "B", "C", "dt", "dA_cumsum", "initial_states"))
    want_out, want_fin = oracle.fused_ref(d["B"], d["x"], d["dt"], d["dA_cumsum"], initial_states=d["initial_states"])
    want_y = oracle.chunk_scan_states_ref(d["C"], want_out, d["dA_cumsum"])
    from ssd_amd import ops as impl
    for limit, chain in ((impl._STATES_ROOM_BYTES, 0), (1 << 20, 1)):
        monkeypatch.setattr(impl, "_STATES_ROOM_BYTES", limit)
        for bf16 in (True, False):
            ops.release_workspaces()
            out, fin = ops._fused_chunk_state_state_passing_fwd(B if bf16 else B.half(), x if bf16 else x.half(), dt, dA,
                                                                torch.bfloat16 if bf16 else torch.float16, initial_states=init)
            torch.cuda.synchronize()
            assert max((k.epochs.last for k in impl._WORKSPACES.values()), default=0) == (chain if bf16 else 0)
            torch.testing.assert_close(out.float().cpu(), want_out, rtol=2.0 ** -7 if bf16 else 2e-3, atol=1e-3)
            torch.testing.assert_close(fin.cpu(), want_fin, rtol=2e-3, atol=1e-3)
        ops.release_workspaces()
        none, fin, y = ops._fused_chunk_state_state_passing_scan_fwd(B, x, C, dt, dA, initial_states=init, return_states=False,
                                                                     y_dtype=torch.float32)
        torch.cuda.synchronize()
        assert none is None and max((k.epochs.last for k in impl._WORKSPACES.values()), default=0) == chain
        assert ops.fused_status() == 0
        torch.testing.assert_close(fin.cpu(), want_fin, rtol=2e-3, atol=1e-3)
        torch.testing.assert_close(y.cpu(), want_y, rtol=2e-3, atol=1e-3)


@pytest.mark.parametrize("kw,dtype", [(dict(L=8192, H=8), "bf16"), (dict(L=2048, H=8, nseq=3), "bf16"), (dict(L=3001, H=6, P=48, N=40, Q=100), "fp16")])
def test_the_calls_in_one_equal_the_calls_one_by_one(ops, oracle, kw, dtype):
    # dt preparation + fused call, and fused call + scan's state half with the passed states wanted in 16 bits: the very
    # kernels of the separate calls, also where those lend the fused call room for the chunk states
    args = dict(b=1, G=1, init=True, dtype=dtype)
    args.update(kw)
    d = oracle.make_inputs(1, **args)
    mv = lambda t: None if t is None else t.cuda()  # noqa: E731
    x, B, C, dt, dA, init, seq = (mv(d[k]) for k in ("x", "B", "C", "dt", "dA_cumsum", "initial_states", "seq_idx"))
    raw = dt.flatten(2).transpose(1, 2)[:, :x.shape[1]].contiguous()
    A = -torch.rand(x.shape[2], device="cuda")
    Q = dt.shape[-1]
    for out_dtype in (x.dtype, torch.float32):
        dA1, dt1 = ops._chunk_cumsum_fwd(raw, A, Q)
        out1, fin1 = ops._fused_chunk_state_state_passing_fwd(B, x, dt1, dA1, out_dtype, initial_states=init, seq_idx=seq)
        out, fin, dA2, dt2 = ops._fused_cumsum_chunk_state_state_passing_fwd(B, x, raw, A, Q, out_dtype, initial_states=init, seq_idx=seq)
        assert out.dtype == out_dtype
        for got, want in ((dA2, dA1), (dt2, dt1), (out, out1), (fin, fin1)):
            assert torch.equal(got, want)
        y1 = ops._chunk_scan_states_fwd(C, out1, dA1, seq_idx=seq)
        out, fin, y = ops._fused_chunk_state_state_passing_scan_fwd(B, x, C, dt1, dA1, out_dtype, initial_states=init, seq_idx=seq)
        assert torch.equal(out, out1) and torch.equal(fin, fin1) and torch.equal(y, y1)
        half = torch.full_like(y, 0.25)
        _, _, y2 = ops._fused_chunk_state_state_passing_scan_fwd(B, x, C, dt1, dA1, out_dtype, initial_states=init, seq_idx=seq, y=half,
                                                                 accumulate=True)
        want = ops._chunk_scan_states_fwd(C, out1, dA1, seq_idx=seq, out=torch.full_like(y, 0.25), accumulate=True)
        assert y2 is half and torch.equal(y2, want)
