"""The scan's state half on the fp32 matrix instructions (every element type, size and alignment the bf16 kernels do not take)
at the edges of its tiles -- 16 or 64 tokens, 1 .. 4 blocks of 16 headdim rows, steps of 16 dstate columns -- against the
oracle, with fp32 sums on both sides."""
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


@pytest.mark.parametrize("c_type,s_type", [("fp32", "fp32"), ("fp16", "fp16"), ("fp32", "fp16"), ("fp16", "fp32"), ("bf16", "fp16"), ("fp16", "bf16")])
@pytest.mark.parametrize("b,L,H,P,N,G,Q,nseq", [
    (1, 1, 1, 1, 1, 1, 1, 0), (2, 70, 3, 16, 16, 1, 64, 0), (1, 130, 2, 17, 15, 2, 65, 3), (1, 300, 4, 40, 24, 2, 100, 0),
    (2, 515, 5, 64, 128, 1, 256, 4), (1, 200, 2, 65, 33, 1, 48, 0), (1, 128, 3, 96, 17, 1, 128, 2), (1, 33, 2, 128, 64, 1, 16, 0),
    (9, 512, 40, 31, 20, 1, 128, 0),              # more tiles than SIMDs: 64 tokens a wave
])
def test_scan_any(ops, oracle, c_type, s_type, b, L, H, P, N, G, Q, nseq):
    types = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
    g = torch.Generator().manual_seed(L * 131 + P)
    nchunks = -(-L // Q)
    C = torch.randn(b, L, G, N, generator=g).to(types[c_type])
    prev = torch.randn(b, nchunks, H, P, N, generator=g).to(types[s_type])
    dA = -torch.rand(b, H, nchunks, Q, generator=g).cumsum(-1) * 0.05
    seq = torch.randint(0, max(nseq, 1), (b, L), generator=g, dtype=torch.int32).sort(dim=1).values if nseq else None
    want = oracle.chunk_scan_states_ref(C.float(), prev.float(), dA, seq_idx=seq)
    print(f"[scan any] {c_type} {s_type} {(b, L, H, P, N, G, Q, nseq)}", flush=True)
    mv = lambda t: None if t is None else t.cuda()  # noqa: E731
    # products of N terms summed in fp32 in two orders: N * 2^-24 of the sum of their magnitudes (about N here) at most
    tol = dict(rtol=1e-5, atol=max(N, 4) * N * 2.0 ** -22)
    y = ops._chunk_scan_states_fwd(mv(C), mv(prev), mv(dA), seq_idx=mv(seq), out_dtype=torch.float32)
    torch.testing.assert_close(y.cpu(), want, **tol)
    # out of wider rows at odd offsets, into a strided y that is added to
    Cw = torch.randn(b, L, G * N + 3).to(C.dtype).cuda()[..., 1:-2].unflatten(-1, (G, N))
    Cw.copy_(C)
    pw = torch.randn(b, nchunks, H, P, N + 1).to(prev.dtype).cuda()[..., 1:]
    pw.copy_(prev)
    out = torch.full((b, L, H * P + 1), 0.5, device="cuda")
    yv = out[..., 1:].unflatten(-1, (H, P))
    assert ops._chunk_scan_states_fwd(Cw, pw, mv(dA), seq_idx=mv(seq), out=yv, accumulate=True) is yv
    assert torch.equal(yv, y + 0.5) and bool((out[..., 0] == 0.5).all())
    for dtype in (torch.float16, torch.bfloat16):
        assert torch.equal(ops._chunk_scan_states_fwd(mv(C), mv(prev), mv(dA), seq_idx=mv(seq), out_dtype=dtype), y.to(dtype))


def test_more_waves_than_one_launch_holds(ops):
    # chunks of one token: a wave per (token, head), 2^26 of them and some; the state that enters a chunk is its only factor
    L, H = (1 << 20) + 3, 64
    g = torch.Generator(device="cuda").manual_seed(5)
    C = torch.randn(1, L, 1, 1, generator=g, device="cuda")
    prev = torch.randn(1, L, H, 1, 1, generator=g, device="cuda")
    dA = torch.zeros(1, H, L, 1, device="cuda")
    print("[scan any] 2^26 waves", flush=True)
    y = ops._chunk_scan_states_fwd(C, prev, dA)
    assert torch.equal(y, C[:, :, 0, :, None] * prev[..., 0])          # one product each: rounded once
