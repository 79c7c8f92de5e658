"""A wrapper's ordinary call in one (csrc/ssd_host.cpp: *_call) against its general way: the same bits wherever both take the
arguments, and everything out of the ordinary left to the general way -- with its results and its errors."""
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


@pytest.fixture
def both(monkeypatch):
    """both(call) -> (the call as it is, the call the general way, whether the first was done in one)"""
    from ssd_amd import ops as impl
    one = impl._ordinary

    def run(call):
        taken = []
        monkeypatch.setattr(impl, "_ordinary", lambda *a: (taken.append(one(*a)), taken[-1])[1])
        got = call()
        monkeypatch.setattr(impl, "_ordinary", lambda *a: None)
        want = call()
        monkeypatch.setattr(impl, "_ordinary", one)
        return got, want, taken and taken[0] is not None
    return run


def _same(got, want):
    got, want = (v if isinstance(v, tuple) else (v,) for v in (got, want))
    assert len(got) == len(want)
    for a, b in zip(got, want):
        assert a.shape == b.shape and a.dtype == b.dtype and a.device == b.device and a.stride() == b.stride() and not a.requires_grad
        assert torch.equal(a, b)


@pytest.mark.parametrize("kw,out,one", [
    (dict(L=700, H=3, dtype="bf16"), torch.bfloat16, True), (dict(L=700, H=3, dtype="fp16", nseq=3, init=True), torch.float32, True),
    (dict(L=700, H=3, P=40, N=24, Q=100, dtype="fp32", init=True), None, True), (dict(b=2, L=2048, H=24), torch.float32, True),
    (dict(L=2048, H=24, nseq=3), torch.bfloat16, False),             # room for chunk states
    (dict(L=8192, H=80), torch.float32, False),                      # the chain kernel
], ids=str)
def test_equal_to_the_general_way(ops, oracle, both, kw, out, one):
    args = dict(b=1, P=64, N=128, G=1, Q=256)
    args.update(kw)
    d = oracle.make_inputs(1, **args)
    mv = lambda t: None if t is None else t.cuda()  # noqa: E731
    x, B, C, dt, dA, seq, init = (mv(d.get(k)) for k in ("x", "B", "C", "dt", "dA_cumsum", "seq_idx", "initial_states"))
    print(f"[ordinary] {kw}", flush=True)
    got, want, taken = both(lambda: ops._fused_chunk_state_state_passing_fwd_concurrent(B, x, dt, dA, out, initial_states=init, seq_idx=seq))
    _same(got, want)
    assert bool(taken) == one
    for f32 in (True, False):
        got, want, taken = both(lambda: ops._chunk_state_fwd(B, x, dt, dA, seq_idx=seq, states_in_fp32=f32))
        _same(got, want)
        assert taken
    states = ops._chunk_state_fwd(B, x, dt, dA, seq_idx=seq)
    flat = None if init is None else init.flatten(-2)
    for o in (None, torch.bfloat16):
        got, want, taken = both(lambda: ops._state_passing_fwd(states.flatten(-2), dA[..., -1], initial_states=flat, seq_idx=seq,
                                                               chunk_size=dt.shape[-1], out_dtype=o))
        _same(got, want)
        assert taken
    for o in (None, torch.float32):
        got, want, taken = both(lambda: ops._chunk_scan_states_fwd(C, states, dA, seq_idx=seq, out_dtype=o))
        _same(got, want)
        assert taken
    raw, A = torch.randn(x.shape[:3], device="cuda").to(x.dtype), -torch.rand(x.shape[2], device="cuda")
    for bias in (None, torch.randn(x.shape[2], device="cuda")):
        got, want, taken = both(lambda: ops._chunk_cumsum_fwd(raw, A, dt.shape[-1], dt_bias=bias, dt_softplus=True, dt_limit=(0.01, 0.5)))
        _same(got, want)
        assert taken


def test_out_of_the_ordinary(ops, oracle, both):
    d = oracle.make_inputs(1, b=2, L=600, H=4, P=64, N=128, G=1, Q=256, init=True, nseq=3)
    x, B, C, dt, dA, seq, init = (d[k].cuda() for k in ("x", "B", "C", "dt", "dA_cumsum", "seq_idx", "initial_states"))
    fused = lambda B=B, x=x, dt=dt, dA=dA, o=torch.float32, **kw: (  # noqa: E731
        lambda: ops._fused_chunk_state_state_passing_fwd_globalbar(B, x, dt, dA, o, **dict(dict(initial_states=init, seq_idx=seq), **kw)))
    # types and layouts that the general way converts
    for call in (fused(dt=dt.double()), fused(dA=dA.half().double()), fused(seq_idx=seq.long()), fused(B=B.float()),
                 fused(x=x.transpose(2, 3).contiguous().transpose(2, 3)), fused(x=torch.nn.Parameter(x, requires_grad=False)),
                 fused(initial_states=init.transpose(2, 3).contiguous().transpose(2, 3)),
                 lambda: ops._chunk_scan_states_fwd(C, ops._chunk_state_fwd(B, x, dt, dA), dA.double())):
        got, want, _ = both(call)
        _same(got, want)
    # strides that need no conversion; a gradient asked for (neither way gives one)
    wide = torch.randn(2, 600, 4 * 64 + 16, device="cuda").to(x.dtype)
    xv = wide[..., 8:-8].unflatten(-1, (4, 64))
    xv.copy_(x)
    for call in (fused(x=xv), fused(dt=dt.transpose(1, 2).contiguous().transpose(1, 2)), fused(initial_states=init.half()),
                 fused(initial_states=init.clone().requires_grad_(True))):
        got, want, taken = both(call)
        _same(got, want)
        assert taken
    # errors are the general way's
    for call, error in ((fused(x=x[:, :-1]), AssertionError), (fused(seq_idx=seq[:1]), AssertionError), (fused(initial_states=init[:1]), AssertionError),
                        (fused(dt=dt[..., :-1]), AssertionError), (fused(x=x.double(), B=B.double()), TypeError),
                        (fused(x=x.cpu(), B=B.cpu()), RuntimeError), (lambda: ops._chunk_cumsum_fwd(dt[:, :, 0].transpose(1, 2), dA[0, :3, 0, 0], 256), AssertionError),
                        (lambda: ops._state_passing_fwd(init[:, None].flatten(-2), dA[..., 0], seq_idx=seq), AssertionError)):
        with pytest.raises(error):
            call()
    # a stream of the caller's, a captured call
    st = torch.cuda.Stream()
    want = fused()()
    st.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(st):
        got = fused()()
    st.synchronize()
    _same(got, want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = fused()()
    for _ in range(3):
        got[0].zero_()
        graph.replay()
        torch.cuda.synchronize()
        _same(got, want)


def test_no_memory_is_torchs_own_error(ops):
    # outputs of 4 TiB and more over inputs of a few elements: no kernel is launched
    b, L, H, P, N = 1, 1 << 20, 128, 64, 128
    one = lambda *shape, dtype=torch.float32: torch.zeros((1,) * (len(shape) - 1) + shape[-1:], dtype=dtype, device="cuda").expand(shape)  # noqa: E731
    x, B, dt, states = one(b, L, H, P, dtype=torch.bfloat16), one(b, L, 1, N, dtype=torch.bfloat16), one(b, H, L, 1), one(b, L, H, P * N)
    few = dict(x=one(1, 1 << 16, 8, 64, dtype=torch.bfloat16), B=one(1, 1 << 16, 1, 1 << 26, dtype=torch.bfloat16), dt=one(1, 8, 64, 1 << 10))
    for call in (lambda: ops._chunk_state_fwd(B, x, dt, dt), lambda: ops._state_passing_fwd(states, one(b, H, L)),
                 lambda: ops._chunk_cumsum_fwd(one(b, 1 << 30, 1 << 10), one(1 << 10), 256),
                 lambda: ops._chunk_scan_states_fwd(one(1, 1 << 30, 1, 64), one(1, 1 << 22, 64, 64, 64), one(1, 64, 1 << 22, 256), out_dtype=torch.float32),
                 lambda: ops._fused_chunk_state_state_passing_fwd(few["B"], few["x"], few["dt"], few["dt"], torch.float32)):
        with pytest.raises(torch.OutOfMemoryError):
            call()
    torch.cuda.empty_cache()
