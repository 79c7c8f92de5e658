"""The stand-alone recurrence around its groups of 4 / 8 / 16 chunks in flight and its windows of 64 decays: chunk counts
on both sides of each, with and without sequence starts, in place, and on planes that are no multiple of four."""
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


@pytest.mark.parametrize("chunks", [1, 2, 4, 5, 15, 16, 17, 31, 63, 64, 65, 80, 127, 128, 129, 200])
@pytest.mark.parametrize("heads,dim", [(3, 260), (2, 7), (70, 4096)])
@pytest.mark.parametrize("packed", [False, True])
def test_recurrence_around_its_groups_and_windows(ops, chunks, heads, dim, packed):
    g = torch.Generator().manual_seed(chunks * 7 + dim)
    b, Q = 1, 16
    states = torch.randn(b, chunks, heads, dim, generator=g)
    da = -torch.rand(b, heads, chunks, generator=g)
    init = torch.randn(b, heads, dim, generator=g)
    seq = torch.cumsum((torch.rand(b, chunks * Q - 3, generator=g) < 0.02).int(), dim=1, dtype=torch.int32) if packed else None
    print(f"[passing] C={chunks} H={heads} dim={dim} packed={packed}", flush=True)
    s, before, want = init.double(), torch.zeros(b, dtype=torch.int32), []
    for c in range(chunks):
        want.append(s)
        last = before if seq is None else seq[:, min((c + 1) * Q, seq.shape[1]) - 1]
        s = (torch.exp(da[:, :, c].double()) * (last == before)[:, None])[..., None] * s + states[:, c].double()
        before = last
    want = torch.stack(want, dim=1)
    out, fin = ops._state_passing_fwd(states.cuda(), da.cuda(), initial_states=init.cuda(), seq_idx=None if seq is None else seq.cuda(),
                                      chunk_size=Q)
    # one rounding of the product and the sum each per chunk and 2^-21 for the exponential; the decay makes a geometric
    # sum of at most 1 / (1 - mean decay) of them
    tol = dict(rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(out.cpu().double(), want, **tol)
    torch.testing.assert_close(fin.cpu().double(), s, **tol)


@pytest.mark.parametrize("chunks", [5, 20, 80])            # four, eight and sixteen chunks in flight
@pytest.mark.parametrize("dim,gap", [(260, 0), (260, 12), (260, 3), (7, 2)])     # planes apart: 4-element loads, then single ones
@pytest.mark.parametrize("dtype,out_dtype", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32), (torch.float32, torch.float16)])
def test_recurrence_over_16_bit_and_strided_planes(ops, chunks, dim, gap, dtype, out_dtype):
    g = torch.Generator().manual_seed(chunks + dim)
    b, heads = 2, 3
    wide = torch.randn(b, chunks, heads, dim + gap, generator=g).to(dtype)
    states = wide[..., :dim]
    da = -torch.rand(b, heads, chunks, generator=g)
    init = torch.randn(b, heads, dim + gap, generator=g)[..., :dim]
    s, want = init.double(), []
    for c in range(chunks):
        want.append(s)
        s = torch.exp(da[:, :, c].double())[..., None] * s + states[:, c].double()
    want = torch.stack(want, dim=1)
    out, fin = ops._state_passing_fwd(wide.cuda()[..., :dim], da.cuda(), initial_states=init.cuda(), out_dtype=out_dtype)
    assert out.dtype == out_dtype and fin.dtype == torch.float32
    # the sums are fp32 whatever the planes are stored as; a 16-bit `out` rounds once on its way
    torch.testing.assert_close(fin.cpu().double(), s, rtol=1e-5, atol=1e-5)
    half = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[out_dtype]
    torch.testing.assert_close(out.cpu().double(), want, rtol=1e-5 + half, atol=1e-5)


@pytest.mark.parametrize("L", [16, 64 * 5, 64 * 70 + 1])
def test_in_place_behind_the_chunk_states(ops, oracle, L):
    # fp32 inputs: the chunk states are written into `out` and turned into the passed states there
    d = oracle.make_inputs(1, b=1, L=L, H=2, P=24, N=40, G=1, Q=64, dtype="fp32", nseq=0, init=True)
    want_out, want_fin = oracle.fused_ref(d["B"], d["x"], d["dt"], d["dA_cumsum"], initial_states=d["initial_states"])
    out, fin = ops._fused_chunk_state_state_passing_fwd(d["B"].cuda(), d["x"].cuda(), d["dt"].cuda(), d["dA_cumsum"].cuda(), torch.float32,
                                                        initial_states=d["initial_states"].cuda())
    torch.testing.assert_close(out.cpu(), want_out, rtol=1e-4, atol=1e-4)
    torch.testing.assert_close(fin.cpu(), want_fin, rtol=1e-4, atol=1e-4)
