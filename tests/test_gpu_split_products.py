"""Chunk states of fp32, fp16 and odd-sized inputs as products of bf16 parts: the error against 64 bits stays that of fp32
sums, whatever the magnitudes, at the edges of steps (32 tokens), quarters and tiles; what is not finite goes the fp32 way."""
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


def _exact(x, B, dt, dA, Q):
    b, L, H, P = x.shape
    out = []
    for c in range(-(-L // Q)):
        t0, t1 = c * Q, min(L, c * Q + Q)
        w = torch.exp(torch.clamp(dA[:, :, c, -1:].double() - dA[:, :, c, :t1 - t0].double(), max=0.0)) * dt[:, :, c, :t1 - t0].double()
        xw = (x[:, t0:t1].double().permute(0, 2, 3, 1) * w[:, :, None]).contiguous()
        out.append(torch.matmul(xw, B[:, t0:t1].double().repeat_interleave(H // B.shape[2], 2).transpose(1, 2).contiguous()))
    return torch.stack(out, 1)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=str)
@pytest.mark.parametrize("L,Q", [(1, 40), (31, 40), (33, 40), (95, 40), (127, 127), (129, 129), (200, 100), (515, 257), (700, 300), (1700, 100)])
@pytest.mark.parametrize("P,N,H", [(20, 24, 2), (65, 17, 3), (64, 96, 40)])
def test_error_is_that_of_fp32_sums(ops, dtype, L, Q, P, N, H):
    g = torch.Generator().manual_seed(L + P)
    C = -(-L // Q)
    # magnitudes over twelve (f16: six) orders beside each other
    spread = lambda *s: (torch.randn(s, generator=g) * 10.0 ** (torch.rand(s, generator=g) * (6 if dtype == torch.float16 else 12) - 4)).to(dtype)  # noqa: E731
    dt, dA = torch.rand(1, H, C, Q, generator=g), -torch.rand(1, H, C, Q, generator=g).cumsum(-1) * 0.05
    for make in (spread, lambda *s: torch.randn(s, generator=g).to(dtype)):
        x, B = make(1, L, H, P), make(1, L, 1, N)
        got = ops._chunk_state_fwd(B.cuda(), x.cuda(), dt.cuda(), dA.cuda())
        want = _exact(x, B, dt, dA, Q)
        # weights and products rounded to fp32 (exp's argument included: |dA| up to 7), L sums of them; too wide to see a product of
        # parts left out, which is test_every_product_of_parts_counts
        bound = torch.matmul(x.double().abs().permute(0, 2, 3, 1), B.double().abs().transpose(1, 2).contiguous()).amax()
        err = (got.double().cpu() - want)
        assert float(err.norm() / want.norm()) < 4e-6 and float(err.abs().amax()) <= 2e-5 * float(bound)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=str)
def test_what_is_not_finite_stays_where_it_is(ops, dtype):
    L, Q, H, P, N = 300, 100, 3, 40, 24
    g = torch.Generator().manual_seed(3)
    x, B = torch.randn(1, L, H, P, generator=g).to(dtype), torch.randn(1, L, 1, N, generator=g).to(dtype)
    dt, dA = torch.rand(1, H, 3, Q, generator=g) + 0.1, -torch.rand(1, H, 3, Q, generator=g).cumsum(-1) * 0.05
    clean = ops._chunk_state_fwd(B.cuda(), x.cuda(), dt.cuda(), dA.cuda())
    x[0, 100, 1, 7], x[0, 230, 2, 11] = float("inf"), float("nan")        # the first token of a chunk too: what padding reads
    B[0, 20, 0, 5] = -float("inf")
    got = ops._chunk_state_fwd(B.cuda(), x.cuda(), dt.cuda(), dA.cuda())
    assert bool((got[0, 1, 1, 7].isinf() & (got[0, 1, 1, 7].sign() == B[0, 100, 0].sign().cuda())).all())
    assert bool(got[0, 2, 2, 11].isnan().all()) and bool(got[0, 0, :, :, 5].isinf().all())
    got[0, 1, 1, 7], got[0, 2, 2, 11], got[0, 0, :, :, 5] = clean[0, 1, 1, 7], clean[0, 2, 2, 11], clean[0, 0, :, :, 5]
    torch.testing.assert_close(got, clean, rtol=1e-5, atol=1e-5)
    if dtype == torch.float32:        # rounds to an infinite bf16, is none
        x, B = torch.full((1, 1, 1, 2), 3.4e38), torch.full((1, 1, 1, 2), 0.5)
        one = ops._chunk_state_fwd(B.cuda(), x.cuda(), torch.ones(1, 1, 1, 1, device="cuda"), torch.zeros(1, 1, 1, 1, device="cuda"))
        torch.testing.assert_close(one.cpu(), torch.full((1, 1, 1, 2, 2), 1.7e38))


# Sizes that run the products of parts (tests/test_generic_way_cpu.py holds the rule to them): tiles of 64 x 64, 64 x 32, 48 x 48 and
# smaller ones, a quarter of a chunk or a whole one per wave, ragged last chunks, odd edges.
PARTS_FP32 = [(515, 257, 64, 128, 70), (300, 257, 64, 128, 33), (300, 257, 63, 127, 2), (700, 100, 64, 128, 80), (1510, 100, 48, 63, 90), (2300, 100, 48, 40, 90)]
PARTS_16 = [(515, 257, 64, 64, 90), (300, 257, 31, 63, 2), (700, 64, 64, 63, 100), (2300, 100, 32, 63, 90), (700, 100, 64, 63, 110)]
PARTS = [(torch.float32, *v) for v in PARTS_FP32] + [(t, *v) for t in (torch.float16, torch.bfloat16) for v in PARTS_16]


@pytest.mark.parametrize("dtype,L,Q,P,N,H", PARTS, ids=str)
def test_every_product_of_parts_counts(ops, dtype, L, Q, P, N, H):
    # Weights that are powers of two, so that nothing but the products and their sums rounds: measured 0.5e-7 of the norm, and 1.3e-6
    # or more with one of the products of parts left out.  The weights reach to where a third bf16 part would be subnormal and to
    # where the sums would be infinite on their way (the fp32 instructions then); so does an fp32 B.
    g = torch.Generator(device="cuda").manual_seed(L + P)
    C = -(-L // Q)
    x = torch.randn(1, L, H, P, generator=g, device="cuda").to(dtype)
    B = torch.randn(1, L, 1, N, generator=g, device="cuda").to(dtype)
    dA = torch.zeros(1, H, C, Q, device="cuda")
    for e, e_B in ((0, 0), (-118, 0), (106, 0)) + (((0, -118), (0, 106), (60, -118)) if dtype == torch.float32 else ()):
        dt, Bs = torch.full((1, H, C, Q), 2.0 ** e, device="cuda"), B * 2.0 ** e_B
        print(f"[parts] {dtype} {(L, Q, P, N, H)} 2^{e} 2^{e_B}", flush=True)
        got = ops._chunk_state_fwd(Bs, x, dt, dA)
        want = _exact(x, Bs, dt, dA, Q)
        err = float((got.double() - want).norm() / want.norm())
        assert err < 4e-7, (e, e_B, err)


@pytest.mark.parametrize("dtype,L,Q,P,N,H", PARTS, ids=str)
def test_what_is_not_finite_stays_where_it_is_on_every_tile(ops, dtype, L, Q, P, N, H):
    g = torch.Generator(device="cuda").manual_seed(L + P)
    C = -(-L // Q)
    x = torch.randn(1, L, H, P, generator=g, device="cuda").to(dtype)
    B = torch.randn(1, L, 1, N, generator=g, device="cuda").to(dtype)
    dt = torch.rand(1, H, C, Q, generator=g, device="cuda") + 0.1
    dA = -torch.rand(1, H, C, Q, generator=g, device="cuda").cumsum(-1) * 0.05
    clean = ops._chunk_state_fwd(B, x, dt, dA)
    last = (C - 1) * Q                                    # the last chunk's first token: what padding reads
    x[0, last, 1, P - 1], x[0, Q - 1, 0, 3], B[0, Q // 2, 0, N - 1] = float("inf"), float("nan"), -float("inf")
    print(f"[parts not finite] {dtype} {(L, Q, P, N, H)}", flush=True)
    got = ops._chunk_state_fwd(B, x, dt, dA)
    assert bool((got[0, C - 1, 1, P - 1].isinf() & (got[0, C - 1, 1, P - 1].sign() == B[0, last, 0].sign())).all())
    assert bool(got[0, 0, 0, 3].isnan().all()) and bool(got[0, 0, 1:, :, N - 1].isinf().all())
    for at in ((0, C - 1, 1, P - 1), (0, 0, 0, 3), (0, 0, slice(None), slice(None), N - 1)):
        got[at] = clean[at]
    # sums of up to Q products in two orders: Q 2^-24 of their magnitudes, which are of order one, at most
    torch.testing.assert_close(got, clean, rtol=1e-5, atol=Q * 2.0 ** -22)
