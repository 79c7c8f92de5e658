"""When a wrapper lends the fused call a place for fp32 chunk states: the library's answer for the very tensors of a call
(host logic only, the tensors' memory is not touched)."""
import pytest
import torch

import ssd_amd as ops
from ssd_amd import _lib


def _wants(b=1, L=4096, H=8, P=64, N=128, G=1, Q=256, dtype=torch.bfloat16, out=torch.bfloat16, init=None, x=None, seq=None):
    C = -(-L // Q)
    x = torch.empty(b, L, H, P, dtype=dtype) if x is None else x
    dt = torch.empty(b, H, C, Q)
    out = None if out is None else torch.empty(b, C, H, P, N, dtype=out)
    return _lib.host().wants_states(x, torch.empty(b, L, G, N, dtype=dtype), dt, dt, seq, init, out, torch.empty(b, H, P, N))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_what_the_call_would_run_decides(dtype):
    # 8 heads x 16 chunks: chunk states + recurrence, with a place for the chunk states, on the bf16 kernels and on the
    # fp32 matrix kernel
    assert _wants(dtype=dtype, out=dtype) and _wants(dtype=dtype, out=None)
    assert not _wants(dtype=dtype, out=torch.float32)                       # `out` is such a place
    assert not _wants(dtype=dtype, out=dtype, L=768)                        # three chunks: the walk
    init = torch.empty(1, 8, 64, 128)
    assert _wants(dtype=dtype, out=dtype, init=init)
    # planes that are not one row (a slice of a wider cache): the recurrence cannot walk them, so the call would run on the
    # kernels that walk a sequence and write the chunk states beside it
    sliced = torch.empty(1, 8, 64, 160)[..., :128]
    assert not _wants(dtype=dtype, out=dtype, init=sliced) and not _wants(dtype=dtype, out=None, init=sliced)
    # a batch or head stride is no matter
    assert _wants(dtype=dtype, out=dtype, init=torch.empty(1, 16, 64, 128)[:, ::2])
    old = ops.set_token_split(4)                                            # a kernel is forced: no chunk states wanted
    try:
        assert not _wants(dtype=dtype, out=dtype)
    finally:
        ops.set_token_split(old)


def test_views_off_the_bf16_tiling_are_the_fp32_kernels_business():
    # 384 state tiles of 64 x 64 are its line; an odd token stride keeps bf16 x off the bf16 kernels
    assert _wants(b=4, L=3072, H=48, dtype=torch.float16, out=torch.float16)
    assert not _wants(b=8, L=1024, H=48, dtype=torch.float16, out=torch.float16)
    odd = torch.empty(4, 3072, 48 * 64 + 1, dtype=torch.bfloat16)[..., :48 * 64].unflatten(-1, (48, 64))
    assert _wants(b=4, L=3072, H=48, x=odd) and not _wants(b=4, L=3072, H=48)


def test_arguments_the_call_rejects_are_left_to_it():
    assert not _wants(H=9, G=2, L=1024)
    assert not _wants(x=torch.empty(1, 4096, 64, 8, dtype=torch.bfloat16).transpose(2, 3))
    with pytest.raises(TypeError):
        _wants(dtype=torch.float64)


@pytest.mark.parametrize("chunks,H,seq,want,scan", [
    (88, 4, True, True, True), (89, 4, True, False, True), (122, 4, True, False, True), (123, 4, True, False, False), (123, 4, False, True, True),
    (79, 8, True, True, True), (80, 8, True, False, False), (80, 8, False, True, True),
    (47, 16, True, True, True), (48, 16, True, True, False), (65, 16, True, True, False), (66, 16, True, False, False), (66, 16, False, True, True),
    (33, 24, True, True, True), (34, 24, True, True, False), (56, 24, True, True, False), (57, 24, True, False, False), (57, 24, False, True, True),
    (17, 48, True, True, True), (18, 48, True, True, False), (31, 48, True, True, False), (32, 48, False, False, False),     # few no more
    (512, 8, True, False, False), (512, 8, False, True, True),                      # long enough for the pair at any number of units
])
def test_packed_sequences_keep_the_chain_kernel_where_its_chains_are_cut(chunks, H, seq, want, scan):
    # chunks of 256 tokens, dstate 128; want: bf16 `out`, scan: the call without passed states
    L = chunks * 256
    seq = torch.zeros(1, L, dtype=torch.int32) if seq else None
    assert _wants(L=L, H=H, seq=seq) == want and _wants(L=L, H=H, seq=seq, out=None) == scan
    if seq is not None:                                                             # fp16 `out`: not the chain kernel's
        assert _wants(L=L, H=H, seq=seq, out=torch.float16) == (want or chunks == 512)


def test_room_is_bounded_and_a_call_does_without_it(monkeypatch):
    from ssd_amd import ops as impl
    x = torch.empty(1)
    assert impl._states_room(x, 1, 16, 8, 64, 128).shape == (1, 16, 8, 64, 128)
    def full(*args, **kw):
        raise torch.OutOfMemoryError("no memory")
    monkeypatch.setattr(impl.torch, "empty", full)
    assert impl._states_room(x, 1, 16, 8, 64, 128) is None                # the memory is not there
    monkeypatch.setattr(impl.torch, "empty", lambda *args, **kw: pytest.fail("more than the bound was asked for"))
    limit = impl._STATES_ROOM_BYTES // (4 * 8 * 64 * 128)
    assert impl._states_room(x, 1, limit + 1, 8, 64, 128) is None


def test_sizes_off_the_bf16_tilings_are_not_the_row_kernels():
    # headdim 48 and 80, chunks of 384, initial states at an odd address: the row kernel could, with 16 bits of x * w where their own
    # kernel has 24, so they keep that one and with a 16-bit out its room for chunk states
    for b, L, H, P, Q in ((1, 65536, 4, 48, 128), (1, 131072, 16, 80, 128), (1, 131072, 2, 64, 384), (1, 4096, 8, 48, 256), (2, 640, 30, 48, 256)):
        for workspace in (False, True):
            assert ops.fused_plan(b, L, H, P, 128, 1, Q, workspace=workspace, compute_units=256)["rows"] == 0
    assert _wants(L=4096, H=8, P=48) and _wants(L=8192, H=2, Q=384) and _wants(b=2, L=4096, H=16, P=80, Q=128)
    assert _wants(b=2, L=2048, H=24, init=torch.empty(2 * 24 * 64 * 128 + 1)[1:].view(2, 24, 64, 128))


@pytest.mark.parametrize("H,chunks,packed,two", [
    (80, 8, True, True), (80, 8, False, True), (80, 9, True, True), (80, 10, True, False), (80, 10, False, True),      # one round: 1.5 unit-chunks a unit
    (160, 4, True, True), (160, 5, True, False), (160, 6, True, False), (160, 6, False, True), (96, 9, True, False), (80, 12, True, False),
    (80, 13, True, True), (160, 8, True, True), (96, 12, True, True), (96, 12, False, True), (104, 12, False, False),  # two rounds
])
def test_scan_without_passed_states_in_two_launches(H, chunks, packed, two):
    seq = torch.zeros(1, 256 * chunks, dtype=torch.int32) if packed else None
    assert _wants(L=256 * chunks, H=H, out=None, seq=seq) == two
