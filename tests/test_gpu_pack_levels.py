"""The prompt pack kernels' level arithmetic on the GPU: the same bytes and scales as the decode
token's kernel, which divides every value by its scale, on ties, extremes, NaN and infinities."""
import pytest
import torch

from layer_quant_amd import _abi

pytestmark = pytest.mark.gpu


def _values(t, d, dtype, gen):
    x = torch.randn(t, d, generator=gen)
    x[0::8] = torch.randint(-14, 15, (len(x[0::8]), d), generator=gen) / 4.0  # ties: 14 quarters = 7 halves
    x[1::8, 3] = 2 * x[1::8, 4]                   # a value that may be half the absmax
    x[2::8] *= 1e-9                               # the 1e-8 scale floor
    x[3::8] *= 3e4
    x[4, 5], x[4, 37], x[12, 70] = float("nan"), float("inf"), float("-inf")
    x[20] = float("nan")
    x[28] = 0.0
    if dtype == torch.float32:
        x[36] *= 1e38
        x[44] *= 1e-39
    return x.to(dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("g", [8, 16, 32, 64, 128])
def test_prompt_levels_equal_token_levels(gpu, dtype, g):
    b, h, t, d = 1, 2, 333, 128
    gen = torch.Generator().manual_seed(g)
    x = torch.stack([_values(t, d, dtype, gen) for _ in range(b * h)]).view(b, h, t, d).to(gpu)

    def cache():
        return (torch.zeros(b, h, t, d // 2, dtype=torch.uint8, device=gpu),
                torch.zeros(b, h, t, d // g, device=gpu))

    prompt, token = cache(), cache()
    _abi.int4_pack_kv(x, *prompt, torch.arange(t, device=gpu), g)
    for i in range(t):  # one token per call: the one-lane-per-byte kernel
        _abi.int4_pack_kv(x[:, :, i:i + 1], *token, torch.tensor([i], device=gpu), g)
    assert torch.equal(prompt[0], token[0])
    assert torch.equal(prompt[1], token[1])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("d,g", [(64, 64), (128, 64), (128, 128), (256, 128), (512, 64)])
@pytest.mark.parametrize("t", [32, 33, 71, 130])
def test_groups_over_several_lanes(gpu, dtype, d, g, t):
    """Groups that span lanes: odd token counts end inside a workgroup, a group's values in one lane
    only (its neighbours zero, NaN or infinite), positions in any order and outside the cache."""
    b, h, cap = 2, 2, t + 3
    gen = torch.Generator().manual_seed(d + g + t)
    x = torch.stack([_values(max(t, 48), d, dtype, gen)[:t] if d > 70 else
                     torch.randn(t, d, generator=gen).to(dtype) for _ in range(b * h)])
    x[:, 5] = 0
    x[:, 5, d - 1] = 3  # the scale comes from the group's last lane
    x[:, 6, : d // 2] = float("inf")
    x = x.view(b, h, t, d).to(gpu)
    pos = torch.randperm(cap, generator=gen)[:t]
    pos[1], pos[2] = -1, cap
    pos = pos.to(gpu)

    def cache():
        return (torch.full((b, h, cap, d // 2), 9, dtype=torch.uint8, device=gpu),
                torch.full((b, h, cap, d // g), -1.0, device=gpu))

    prompt, token = cache(), cache()
    _abi.int4_pack_kv(x, *prompt, pos, g)
    for i in range(t):  # one token per call: the one-lane-per-byte kernel
        _abi.int4_pack_kv(x[:, :, i:i + 1], *token, pos[i:i + 1], g)
    assert torch.equal(prompt[0], token[0])
    assert torch.equal(prompt[1], token[1])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("g", [16, 32, 64, 128])
def test_packed_rows_aligned_to_words_only(gpu, dtype, g):
    """Packed rows 68 bytes apart from an offset of 4: the kernel with 4-byte stores at the group sizes
    that aligned caches take to the one with wide stores. Nothing is written between the rows."""
    b, h, t, d = 1, 2, 77, 128
    gen = torch.Generator().manual_seed(g)
    x = torch.stack([_values(t, d, dtype, gen) for _ in range(b * h)]).view(b, h, t, d).to(gpu)
    pos = torch.arange(t, device=gpu)
    buf = torch.full((4 + b * h * t * 68,), 9, dtype=torch.uint8, device=gpu)
    rows = buf[4:].view(b, h, t, 68)
    token = torch.zeros(b, h, t, d // 2, dtype=torch.uint8, device=gpu)
    scale, token_scale = (torch.zeros(b, h, t, d // g, device=gpu) for _ in range(2))
    _abi.int4_pack_kv(x, rows[..., :d // 2], scale, pos, g)
    for i in range(t):  # one token per call: the one-lane-per-byte kernel
        _abi.int4_pack_kv(x[:, :, i:i + 1], token, token_scale, pos[i:i + 1], g)
    assert torch.equal(rows[..., :d // 2], token)
    assert torch.equal(scale, token_scale)
    assert (buf[:4] == 9).all() and (rows[..., d // 2:] == 9).all()
