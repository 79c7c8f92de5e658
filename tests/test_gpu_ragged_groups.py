"""Groups whose state tiles (32 headdim rows) are no multiple of four: the chunk-state launch of the four-tile kernel with
waves that have no tile of their own, and the fused call as that launch + recurrence."""
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


CASES = [
    dict(b=1, L=700, H=1, P=32),                                    # one tile
    dict(b=2, L=1500, H=3, P=64, nseq=3),                           # a unit and a half, ragged chunk, packed
    dict(b=2, L=900, H=9, P=32, G=3, Q=128),                        # three groups of three tiles
    dict(b=3, L=1024, H=10, P=64, G=2, N=64, nseq=4),               # two groups of ten
    dict(b=1, L=513, H=7, P=96, N=64, Q=128),                       # 21 tiles, one token in the last chunk
]


@pytest.mark.parametrize("kw", CASES, ids=lambda kw: "-".join(f"{k}{v}" for k, v in kw.items()))
def test_ragged_groups(ops, oracle, kw):
    args = dict(N=128, G=1, Q=256, init=True, nseq=0)
    args.update(kw)
    d = oracle.make_inputs(1, **args)
    mv = lambda t: None if t is None else t.cuda()  # noqa: E731
    x, B, dt, dA, init, seq = (mv(d[k]) for k in ("x", "B", "dt", "dA_cumsum", "initial_states", "seq_idx"))
    print(f"[ragged] {kw}", flush=True)
    want = oracle.chunk_state_ref(d["B"], d["x"], d["dt"], d["dA_cumsum"], seq_idx=d["seq_idx"])
    want_out, want_fin = oracle.fused_ref(d["B"], d["x"], d["dt"], d["dA_cumsum"], initial_states=d["initial_states"], seq_idx=d["seq_idx"])
    guard = torch.full((want.numel() + 4096,), 7.0, device="cuda")          # what lies behind the states stays as it is
    states = guard[:want.numel()].view(want.shape)
    old = ops.set_token_split(1)
    try:
        for seg in (0, 1, 3):
            olds = ops.set_segment_chunks(seg)
            try:
                states.fill_(float("nan"))
                assert ops._chunk_state_fwd(B, x, dt, dA, seq_idx=seq, states=states) is states
            finally:
                ops.set_segment_chunks(olds)
            torch.testing.assert_close(states.cpu(), want, rtol=2e-3, atol=1e-3)
            assert bool((guard[want.numel():] == 7.0).all())
        out, fin = ops._fused_chunk_state_state_passing_fwd(B, x, dt, dA, torch.float32, initial_states=init, seq_idx=seq, states=states)
    finally:
        ops.set_token_split(old)
    torch.testing.assert_close(out.cpu(), want_out, rtol=2e-3, atol=1e-3)
    torch.testing.assert_close(fin.cpu(), want_fin, rtol=2e-3, atol=1e-3)
    half = ops._chunk_state_fwd(B, x, dt, dA, seq_idx=seq, states=torch.empty(want.shape, device="cuda", dtype=torch.bfloat16))
    torch.testing.assert_close(half.float().cpu(), want, rtol=2.0 ** -7, atol=1e-3)


# 36 chunks of 25 heads and more: the pair; below the row kernel or the walk
@pytest.mark.parametrize("kw,family", [(dict(b=2, L=9216, H=25), "pair"), (dict(b=3, L=5200, H=9, G=3, Q=128, nseq=4), "pair"),
                                       (dict(b=8, L=700, H=33), "token_split"),
                                       # groups of one, two and three tiles, with chunk states enough to fill the chip
                                       (dict(b=8, L=9000, H=8, P=32, G=8), "pair"), (dict(b=4, L=9000, H=8, G=8), "pair"),
                                       (dict(b=8, L=2500, H=8, P=96, G=8, N=64, Q=128, nseq=3), "token_split")])
def test_calls_left_to_the_library(ops, oracle, kw, family):
    args = dict(P=64, N=128, G=1, Q=256, init=True, nseq=0)
    args.update(kw)
    plan = ops.fused_plan(*(args[k] for k in ("b", "L", "H", "P", "N", "G", "Q")), compute_units=256)
    assert plan["family"] == family, plan
    d = oracle.make_inputs(1, **args)
    mv = lambda t: None if t is None else t.cuda()  # noqa: E731
    x, B, dt, dA, init, seq = (mv(d[k]) for k in ("x", "B", "dt", "dA_cumsum", "initial_states", "seq_idx"))
    print(f"[ragged auto] {kw}", flush=True)
    want_out, want_fin = oracle.fused_ref(d["B"], d["x"], d["dt"], d["dA_cumsum"], initial_states=d["initial_states"], seq_idx=d["seq_idx"])
    states = ops._chunk_state_fwd(B, x, dt, dA, seq_idx=seq)
    torch.testing.assert_close(states.cpu(), oracle.chunk_state_ref(d["B"], d["x"], d["dt"], d["dA_cumsum"], seq_idx=d["seq_idx"]), rtol=2e-3, atol=1e-3)
    given = torch.empty_like(states)
    out, fin = ops._fused_chunk_state_state_passing_fwd(B, x, dt, dA, torch.float32, initial_states=init, seq_idx=seq, states=given)
    torch.testing.assert_close(given, states, rtol=2e-3, atol=1e-3)
    torch.testing.assert_close(out.cpu(), want_out, rtol=2e-3, atol=1e-3)
    for dtype in (torch.float32, torch.bfloat16):
        out, fin = ops._fused_chunk_state_state_passing_fwd(B, x, dt, dA, dtype, initial_states=init, seq_idx=seq)
        torch.testing.assert_close(out.float().cpu(), want_out, rtol=2e-3 if dtype == torch.float32 else 2.0 ** -7, atol=1e-3)
        torch.testing.assert_close(fin.cpu(), want_fin, rtol=2e-3, atol=1e-3)
