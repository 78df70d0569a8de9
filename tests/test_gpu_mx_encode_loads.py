"""The MX encoder's value loads: 16-byte loads of contiguous 16-byte aligned rows (bf16, fp16,
fp32) and element loads of every other layout, bit-exact against the oracle."""
import numpy as np
import pytest
import torch

from layer_quant_amd import _abi
from oracle import mx_state as omx

pytestmark = pytest.mark.gpu


def _view(h, form, device):
    """h [B, H, P, N] on the device with the strides that `form` names."""
    b, nh, p, n = h.shape
    if form == "contiguous":
        return h.to(device)
    if form == "padded":        # rows 16-byte aligned, but not adjacent
        base = torch.zeros(b, nh, p, n + 8, dtype=h.dtype, device=device)[..., :n]
    elif form == "odd rows":    # the second row starts off a 16-byte boundary
        base = torch.zeros(b, nh, p, n + 1, dtype=h.dtype, device=device)[..., :n]
    elif form == "odd base":    # rows aligned to each other, the first one is not
        flat = torch.zeros(b * nh * p * n + 8, dtype=h.dtype, device=device)
        base = flat[1:1 + h.numel()].view(h.shape)
    elif form == "heads swapped":
        base = torch.zeros(b, p, nh, n, dtype=h.dtype, device=device).transpose(1, 2)
    else:                       # d_state not contiguous
        base = torch.zeros(b, nh, n, p, dtype=h.dtype, device=device).transpose(2, 3)
    base.copy_(h)
    return base


@pytest.mark.parametrize("form", ["contiguous", "padded", "odd rows", "odd base", "heads swapped",
                                  "transposed"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("n,fb,mode,layout", [(128, 8, 0, "reference"), (48, 4, 1, "reference"),
                                              (16, 4, 0, "compact"), (256, 8, 3, "compact")])
def test_encode_value_loads(gpu, form, dtype, n, fb, mode, layout):
    shape = (2, 3, 37, n)  # 37 rows: a last workgroup that is partly empty
    gen = torch.Generator().manual_seed(n + fb)
    h = (torch.randn(shape, generator=gen) * torch.exp(torch.randn(*shape[:-1], 1, generator=gen)))
    h[0, 0, 0] = 0.0
    h[0, 0, 1, :2] = torch.tensor([2.0 ** 14, -2.0 ** -14])
    h = h.to(dtype)
    q_bytes = n // 2 if layout == "compact" and fb == 4 else n
    out = (torch.empty(*shape[:3], q_bytes, dtype=torch.uint8 if q_bytes < n else torch.int8, device=gpu),
           torch.empty(*shape[:3], n // 16, dtype=torch.uint8, device=gpu),
           torch.empty(*shape[:3], n // (16 if layout == "compact" else 2), dtype=torch.uint8, device=gpu))
    _abi.mx_encode(_view(h, form, gpu), *out, fb, mode, None, 99, 32)
    ref = omx.mx_encode(h.float().numpy(), fb, mode, seed=99, rng_offset=32)
    if layout == "compact":
        ref = omx.to_compact(*ref, fb)
    for name, got, want in zip("qem", out, ref):
        assert np.array_equal(got.cpu().numpy().view(np.uint8), np.asarray(want).view(np.uint8)), name
