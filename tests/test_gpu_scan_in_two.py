"""The scan call without passed states on few chunks: the fused call into room that the wrapper lends, then the scan's own
kernel, on both sides of the line, and the one-launch kernel on the same inputs, against the oracle."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    import ssd_amd
    return ssd_amd


@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("b,L,H,N,Q,seqs,y_dtype,chain", [
    (1, 40, 8, 64, 128, 0, torch.bfloat16, 0),      # one short chunk
    (2, 322, 8, 128, 256, 0, torch.float32, 0),     # two chunks, the second ragged
    (1, 2048, 40, 128, 256, 3, torch.bfloat16, 0),  # eight chunks, packed
    (1, 2304, 96, 128, 256, 0, torch.bfloat16, 0),  # nine chunks of 48 units, the last with two launches
    (1, 2304, 104, 128, 256, 0, torch.bfloat16, 1), # nine chunks of 52 units: one launch
])
def test_both_sides_of_the_line(ops, oracle, b, L, H, N, Q, seqs, y_dtype, chain, accumulate):
    from ssd_amd import ops as impl
    g = torch.Generator().manual_seed(L + H)
    x, B, C = (torch.randn(b, L, *s, generator=g).to(torch.bfloat16) for s in ((H, 64), (1, N), (1, N)))
    A, dt = -torch.rand(H, generator=g) - 0.5, torch.rand(b, L, H, generator=g) * 0.1
    init = torch.randn(b, H, 64, N, generator=g)
    seq = (torch.arange(L) * seqs // L).to(torch.int32).expand(b, L).contiguous() if seqs else None
    dA, dt = oracle.chunk_cumsum_ref(dt, A, Q)
    args = [t.cuda() for t in (B, x, C, dt, dA)]
    ginit, gseq = init.cuda(), None if seq is None else seq.cuda()
    base = 0.25 if accumulate else 0.0

    def run(**kw):
        y = torch.full((b, L, H, 64), base, dtype=y_dtype, device="cuda") if accumulate else None
        return ops._fused_chunk_state_state_passing_scan_fwd(*args, initial_states=ginit, seq_idx=gseq, return_states=False, y=y,
                                                             accumulate=accumulate, y_dtype=y_dtype, **kw)

    ops.release_workspaces()
    none, fin, y = run()
    torch.cuda.synchronize()
    assert none is None and max((k.epochs.last for k in impl._WORKSPACES.values()), default=0) == chain
    _, fin1, y1 = run(_kernel=1)
    states, want_fin = oracle.fused_ref(B, x, dt, dA, initial_states=init, seq_idx=seq)
    size, fin_size = oracle.fused_ref(B.abs(), x.abs(), dt, dA, initial_states=init.abs(), seq_idx=seq)
    want, size = oracle.chunk_scan_states_ref(C, states, dA, seq) + base, oracle.chunk_scan_states_ref(C.abs(), size, dA, seq) + base
    # roundings to bf16 of 2^-9 each, on terms whose sizes the second pair of results sums: the token's weight and its product
    # with x or B in the states; then the state, the decayed C and y itself
    for got, ref, terms, n in ((fin, want_fin, fin_size, 2), (fin1, want_fin, fin_size, 2), (y, want, size, 5), (y1, want, size, 5)):
        worst = ((got.cpu().double() - ref.double()).abs() / (n * 2.0 ** -9 * terms.double() + 1e-5)).max().item()
        assert worst <= 1, worst
