"""The attention calls' small inputs: the last cache position read back to the host, and the additive
bias of a 2-D keep-mask."""
import ctypes

import pytest
import torch

from layer_quant_amd import _abi
from hybrid_quant import int4_8b_attention as ia


def test_arguments_are_rejected_on_the_cpu():
    from test_abi_cpu import _fake

    lib = _abi.lib()
    pos = _fake((3,), torch.int64)
    assert lib.lq_max_position(pos, None, None) == _abi.LQ_ERR_INVALID_ARG
    assert lib.lq_max_position(pos, ctypes.c_void_p(0x1004), None) == _abi.LQ_ERR_INVALID_ARG
    assert lib.lq_max_position(_fake((0,), torch.int64), ctypes.c_void_p(0x1000), None) == _abi.LQ_ERR_INVALID_ARG
    assert lib.lq_max_position(_fake((3,), torch.int32), ctypes.c_void_p(0x1000), None) == _abi.LQ_ERR_INVALID_ARG
    keep = _fake((2, 5), torch.uint8)
    assert lib.lq_keep_mask_bias(keep, _fake((2, 1, 1, 4), torch.float32), None) == _abi.LQ_ERR_INVALID_ARG
    assert lib.lq_keep_mask_bias(keep, _fake((2, 1, 1, 5), torch.bfloat16), None) == _abi.LQ_ERR_INVALID_ARG
    assert _abi.start_max_position(torch.arange(3)) is None
    assert _abi.start_max_position(None) is None


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 257, 4096, 4097, 65535, 65536])
def test_max_position(gpu, n):
    gen = torch.Generator().manual_seed(n)
    pos = torch.randint(-(1 << 40), 1 << 40, (n,), generator=gen).to(gpu)
    assert _abi.start_max_position(pos).wait() == int(pos.max().item())
    wide = torch.randint(-(1 << 40), -1, (n, 3), generator=gen).to(gpu)[:, 1]  # strided, all negative
    assert _abi.start_max_position(wide).wait() == int(wide.max().item())


@pytest.mark.gpu
@pytest.mark.parametrize("offset", [0, 1])  # 16-byte aligned or not
@pytest.mark.parametrize("n", [1, 2, 3, 511, 512, 513, 2047, 4095, 8193, 16383, 16384, 16385, 65535])
def test_max_position_anywhere(gpu, n, offset):
    buf = torch.full((n + 2,), 1 << 50, dtype=torch.int64, device=gpu)  # neighbours are larger
    pos = buf[offset:offset + n]
    pos.copy_(torch.arange(n, device=gpu) - n)
    for at in {0, n // 2, n - 2, n - 1} - {-1}:
        pos[at] += 1 << 41
        assert _abi.start_max_position(pos).wait() == (1 << 41) + at - n
        pos[at] -= 1 << 41


@pytest.mark.gpu
def test_max_position_follows_its_stream(gpu):
    """The value is the one the positions hold when the stream gets there, on any stream."""
    side = torch.cuda.Stream()
    pos = torch.zeros(100, dtype=torch.int64, device=gpu)
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        for i in range(1, 4):
            torch.cuda._sleep(2_000_000)
            pos.fill_(i)
            pending = _abi.start_max_position(pos)
            pos.fill_(99)
            assert pending.wait() == i
    assert _abi.start_max_position(pos[:0]) is None
    assert _abi.start_max_position(pos.int()) is None
    assert _abi.start_max_position(pos.view(10, 10)) is None
    assert _abi.start_max_position(torch.zeros(_abi.MAX_POSITIONS + 1, dtype=torch.int64, device=gpu)) is None


@pytest.mark.gpu
def test_max_positions_pending_together(gpu):
    """A second read started before the first one's wait (a projection that is itself such a call)
    keeps its own value; the slots are taken again afterwards."""
    pos = [torch.full((n,), n, dtype=torch.int64, device=gpu) for n in (3, 50, 700)]
    for _ in range(3):
        started = [_abi.start_max_position(p) for p in pos]
        assert [s.wait() for s in started] == [3, 50, 700]
    free = _abi._free_slots.by_device[gpu.index or 0]
    held = len(free)
    assert held >= 3
    for _ in range(3):
        assert _abi.start_max_position(pos[0]).wait() == 3
    assert len(free) == held
    assert _abi.start_max_position(torch._neg_view(pos[0])) is None


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bool, torch.uint8, torch.int8, torch.int16, torch.int32,
                                   torch.int64, torch.float16, torch.bfloat16, torch.float32,
                                   torch.float64])
@pytest.mark.parametrize("s", [1, 255, 257, 1000])
def test_keep_mask_bias(gpu, dtype, s):
    """Every mask dtype and layout gives the torch expression's bias (int16 and float64 take it)."""
    gen = torch.Generator().manual_seed(s)
    keep = torch.randint(0, 3, (3, s + 5), generator=gen)
    keep[0] = 0
    keep = (keep * torch.randint(-1, 2, keep.shape, generator=gen)).to(dtype)
    if dtype.is_floating_point:
        keep[1, 0], keep[1, 1], keep[1, 2] = -0.0, float("nan"), 1e-7
    want = ia._decode_attention_mask(keep, 3, s, torch.device("cpu"))
    for mask in (keep.to(gpu), keep.t().contiguous().to(gpu).t(), keep.repeat(1, 2).to(gpu)[:, :s + 5]):
        got = ia._decode_attention_mask(mask, 3, s, gpu)
        assert got.dtype == torch.float32 and torch.equal(got.cpu(), want)
    # a one-row mask broadcasts over the batch, a short one is refused, as before
    row = ia._decode_attention_mask(keep[:1].to(gpu), 3, s, gpu)
    assert torch.equal(row.cpu(), ia._decode_attention_mask(keep[:1], 3, s, torch.device("cpu")))
    if s > 3:
        with pytest.raises(RuntimeError):
            ia._decode_attention_mask(keep[:, :2].to(gpu), 3, s, gpu)


@pytest.mark.gpu
def test_max_position_declines_a_captured_stream(gpu):
    """A host read-back cannot be captured: the caller's .item() then refuses as it always did."""
    pos = torch.arange(4, device=gpu)
    assert _abi.start_max_position(pos).wait() == 3
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        assert _abi.start_max_position(pos) is None
        out = pos + 1
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, pos + 1)
