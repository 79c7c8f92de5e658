"""The row kernel (workgroups of 1 .. 5 slices of 16 state rows, loading and multiplying waves) at the edges of its
tiling: groups that the slices do not divide, heads that straddle workgroups, ragged last chunks and steps, one round and
many, both dstates, every output type, packed sequences, strided inputs -- against the oracle."""
import pytest
import torch

pytestmark = pytest.mark.gpu
ROWS = 4          # SSD_KERNEL_ROWS; chunks_per_item is then the slices per workgroup


@pytest.fixture(scope="module")
def ops():
    import ssd_amd
    from ssd_amd import _lib
    _lib.load()
    assert torch.cuda.is_available(), "these tests need the MI355X"
    return ssd_amd


CASES = [
    dict(b=1, L=128, H=1, Q=128),                                   # one round
    dict(b=2, L=1, H=2),                                            # one token
    dict(b=1, L=300, H=3, init=True),                               # ragged, two chunks
    dict(b=2, L=1280, H=5, P=48, N=64, nseq=4, init=True),          # headdim of three slices, dstate 64
    dict(b=1, L=1500, H=6, P=80, G=2, Q=128, nseq=3, init=True),    # slices straddle heads, grouped B, ragged
    dict(b=3, L=640, H=4, P=16, Q=384),                             # one slice a head: workgroups of up to five heads
    dict(b=1, L=4096, H=10, init=True),                             # many rounds
    dict(b=1, L=2049, H=2, P=128, N=64, Q=128, init=True),          # one token in the last chunk
]


@pytest.mark.parametrize("kr", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("kw", CASES, ids=lambda kw: "-".join(f"{k}{v}" for k, v in kw.items()))
def test_rows_kernel(ops, oracle, kw, kr):
    args = dict(P=64, N=128, G=1, Q=256, init=False, nseq=0)
    args.update(kw)
    d = oracle.make_inputs(1, **args)
    mv = lambda t: None if t is None else t.cuda()  # noqa: E731
    x, B, dt, dA, init, seq = (mv(d[k]) for k in ("x", "B", "dt", "dA_cumsum", "initial_states", "seq_idx"))
    print(f"[rows] {kw} kr={kr}", flush=True)
    run = lambda dtype, x=x, B=B, init=init: ops._fused_chunk_state_state_passing_fwd(  # noqa: E731
        B, x, dt, dA, dtype, initial_states=init, seq_idx=seq, _kernel=ROWS, _chunks_per_item=kr)
    want, want_fin = oracle.fused_ref(d["B"], d["x"], d["dt"], d["dA_cumsum"], initial_states=d["initial_states"], seq_idx=d["seq_idx"])
    out, fin = run(torch.float32)
    torch.testing.assert_close(out.cpu(), want, rtol=2e-3, atol=1e-3)
    torch.testing.assert_close(fin.cpu(), want_fin, rtol=2e-3, atol=1e-3)
    for dtype in (torch.bfloat16, torch.float16):
        out16, fin16 = run(dtype)
        assert torch.equal(out16, out.to(dtype)) and torch.equal(fin16, fin)
    # x and B as views into wider rows, initial states in 16 bits out of a wider cache
    wide = torch.randn(*x.shape[:2], x.shape[2] * x.shape[3] + B.shape[2] * B.shape[3] + 24, device="cuda", dtype=x.dtype)
    xv = wide[..., 8:8 + x.shape[2] * x.shape[3]].unflatten(-1, x.shape[2:])
    Bv = wide[..., 16 + x.shape[2] * x.shape[3]:-8].unflatten(-1, B.shape[2:])
    xv.copy_(x)
    Bv.copy_(B)
    out_v, fin_v = run(torch.float32, x=xv, B=Bv)
    assert torch.equal(out_v, out) and torch.equal(fin_v, fin)
    if init is not None:
        for dtype in (torch.bfloat16, torch.float16):
            cache = torch.zeros(*init.shape[:-1], init.shape[-1] + 3, device="cuda", dtype=dtype)[..., 1:-2]
            cache.copy_(init)
            a, fa = run(torch.float32, init=cache)
            e, fe = run(torch.float32, init=cache.float())
            assert torch.equal(a, e) and torch.equal(fa, fe)


# 128 rows and more to a compute unit, a second round of workgroups, few units, long rows: the other families
@pytest.mark.parametrize("kw,rows", [
    (dict(b=8, L=2048, H=24), 3), (dict(b=1, L=4096, H=80), 2), (dict(b=4, L=2048, H=80), 5), (dict(b=4, L=8192, H=64), 4),
    (dict(b=3, L=1100, H=26, P=128, N=64, G=2), 3),
    (dict(b=8, L=2048, H=48), 0), (dict(b=4, L=8192, H=80), 0), (dict(b=1, L=2048, H=24), 0), (dict(b=2, L=8192, H=48), 0),
    (dict(b=1, L=1024, H=80, P=40), 0), (dict(b=1, L=1024, H=80, Q=64), 0), (dict(b=2, L=640, H=30, P=48), 0), (dict(b=1, L=1000, H=50, Q=384), 0),
], ids=lambda v: "-".join(f"{k}{x}" for k, x in v.items()) if isinstance(v, dict) else str(v))
def test_calls_left_to_the_library(ops, oracle, kw, rows):
    args = dict(P=64, N=128, G=1, Q=256, init=True, nseq=3)
    args.update(kw)
    plan = ops.fused_plan(*(args[k] for k in ("b", "L", "H", "P", "N", "G", "Q")), compute_units=256)
    assert plan["rows"] == rows, plan
    if not rows or args["b"] * args["L"] * args["H"] > 1.1e6:
        return
    d = oracle.make_inputs(1, **args)
    mv = lambda t: None if t is None else t.cuda()  # noqa: E731
    x, B, dt, dA, init, seq = (mv(d[k]) for k in ("x", "B", "dt", "dA_cumsum", "initial_states", "seq_idx"))
    print(f"[rows auto] {kw}", flush=True)
    kw = dict(initial_states=init, seq_idx=seq)
    out, fin = ops._fused_chunk_state_state_passing_fwd(B, x, dt, dA, torch.float32, **kw)
    o, f = ops._fused_chunk_state_state_passing_fwd(B, x, dt, dA, torch.float32, _kernel=ROWS, _chunks_per_item=rows, **kw)
    assert torch.equal(out, o) and torch.equal(fin, f)
    want, want_fin = oracle.fused_ref(d["B"], d["x"], d["dt"], d["dA_cumsum"], initial_states=d["initial_states"], seq_idx=d["seq_idx"])
    torch.testing.assert_close(out.cpu(), want, rtol=2e-3, atol=1e-3)
    torch.testing.assert_close(fin.cpu(), want_fin, rtol=2e-3, atol=1e-3)
    # x with its heads in front of the tokens: not a layout of this kernel, the call runs as before it
    xt = x.transpose(1, 2).contiguous().transpose(1, 2)
    out, fin = ops._fused_chunk_state_state_passing_fwd(B, xt, dt, dA, torch.float32, **kw)
    torch.testing.assert_close(out.cpu(), want, rtol=2e-3, atol=1e-3)
    torch.testing.assert_close(fin.cpu(), want_fin, rtol=2e-3, atol=1e-3)
    # captured: replays between eager calls
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        g_out, g_fin = ops._fused_chunk_state_state_passing_fwd(B, x, dt, dA, torch.float32, **kw)
    for _ in range(3):
        g_out.zero_()
        g_fin.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(g_out, o) and torch.equal(g_fin, f)


# headdim 48 and 80, chunks of 384, initial states at an odd address: not sizes of the other bf16 kernels, the call stays with
# the kernel that multiplies in 24 bits
@pytest.mark.parametrize("kw", [dict(b=2, L=700, H=30, P=48, Q=128), dict(b=1, L=1400, H=40, P=80), dict(b=1, L=1000, H=50, P=64, Q=384),
                                dict(b=4, L=700, H=48, P=64, odd_init=True)], ids=lambda kw: "-".join(f"{k}{v}" for k, v in kw.items()))
def test_sizes_off_the_tilings_keep_their_products(ops, kw):
    args = dict(N=128, Q=256, odd_init=False)
    args.update(kw)
    b, L, H, P, N, Q = (args[k] for k in "bLHPNQ")
    C, g = -(-L // Q), torch.Generator().manual_seed(L)
    x, B = torch.randn(b, L, H, P, generator=g).to(torch.bfloat16), torch.randn(b, L, 1, N, generator=g).to(torch.bfloat16)
    dt, dA = torch.rand(b, H, C, Q, generator=g) + 0.5, -torch.rand(b, H, C, Q, generator=g).cumsum(-1) * 2.0 ** -12
    init = torch.randn(b, H, P, N, generator=g)
    want, state = [], init.double()
    for c in range(C):
        t0, t1 = c * Q, min(L, c * Q + Q)
        want.append(state)
        w = torch.exp(dA[:, :, c, -1:].double() - dA[:, :, c, :t1 - t0].double()) * dt[:, :, c, :t1 - t0].double()
        xw = (x[:, t0:t1].double().permute(0, 2, 3, 1) * w[:, :, None]).contiguous()
        state = torch.exp(dA[:, :, c, -1].double())[..., None, None] * state + torch.matmul(xw, B[:, t0:t1].double().transpose(1, 2).contiguous())
    ginit = torch.empty(b * H * P * N + 1, device="cuda")[1:].view(init.shape) if args["odd_init"] else torch.empty(init.shape, device="cuda")
    ginit.copy_(init)
    print(f"[rows off tilings] {kw}", flush=True)
    out, fin = ops._fused_chunk_state_state_passing_fwd(B.cuda(), x.cuda(), dt.cuda(), dA.cuda(), torch.float32, initial_states=ginit)
    # Sums of up to 384 products one after the other leave sqrt(384 / 2) * 2^-24 / sqrt(3) = 5e-7 of their size, of 32 at a time less;
    # the weights add 1e-7.  x * w in 16 bits alone is at 2^-18 / sqrt(3) = 2e-6.
    for got, ref in ((out, torch.stack(want, 1)), (fin, state)):
        err = float((got.double().cpu() - ref).norm() / ref.norm())
        assert err < 6e-7, err
