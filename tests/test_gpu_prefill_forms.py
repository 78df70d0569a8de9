"""The MFMA prefill's row accesses and key groups: every form of the query and output rows (16-byte
accesses or element accesses) with one and with two key groups, at the edges of the 32-position
blocks, against the float64 oracle."""
import pytest
import torch

from helpers import assert_close_rel
from layer_quant_amd import _abi
from oracle import int4_kv as oik

pytestmark = pytest.mark.gpu


def _rows(x, form, device, dtype):
    """x [B, H, L, D] (None: a NaN-filled output) as rows of the form."""
    b, h, n, d = x.shape
    if form == "contiguous":
        t = torch.full((b, h, n, d), float("nan"), device=device, dtype=dtype)
    elif form == "transposed":    # [B, L, H, D]: 16-byte aligned rows
        t = torch.full((b, n, h, d), float("nan"), device=device, dtype=dtype).transpose(1, 2)
    elif form == "odd rows":      # rows of D + 1 elements
        t = torch.full((b, h, n, d + 1), float("nan"), device=device, dtype=dtype)[..., :d]
    elif form == "odd base":
        t = torch.full((b * h * n * d + 8,), float("nan"), device=device, dtype=dtype)
        t = t[1:1 + b * h * n * d].view(b, h, n, d)
    else:                         # head_dim not contiguous
        t = torch.full((b, h, d, n), float("nan"), device=device, dtype=dtype).transpose(2, 3)
    return t


# (b, hkv, nrep): up to 512 workgroups take two key groups, more take one
GRIDS = {"two groups": [(1, 2, 4), (2, 1, 1), (1, 1, 8), (1, 2, 2)],
         "one group": [(16, 8, 4), (32, 16, 1)]}


@pytest.mark.parametrize("grid", list(GRIDS))
@pytest.mark.parametrize("L", [1, 31, 32, 33, 64, 65, 129, 200])
@pytest.mark.parametrize("qform,oform", [("contiguous", "contiguous"), ("transposed", "odd rows"),
                                         ("odd base", "transposed"), ("columns", "columns")])
def test_prefill_forms(gpu, diag, grid, L, qform, oform):
    diag.set("LQ_PREFILL_REQUIRE_MFMA")
    if grid == "one group":
        # B * Hkv units of ceil(ceil(L / 32) * nrep / 4) workgroups: over 512 from L = 129 (nrep 4)
        L += 100 if L < 129 else 0
    for i, (b, hkv, nrep) in enumerate(GRIDS[grid]):
        g = (32, 64, 128)[(i + L) % 3]
        gen = torch.Generator().manual_seed(1000 * i + L)
        cache = oik.allocate_cache(b, hkv, L + 3, 128, g)
        k, v = (torch.randn(b, hkv, L, 128, generator=gen).to(torch.bfloat16) for _ in range(2))
        oik.pack_kv_into_cache(cache, k, v, torch.arange(L), g)
        q = (torch.randn(b, hkv * nrep, L, 128, generator=gen) * 2).to(torch.bfloat16)
        ref = oik.prefill_attention(q, cache["k_packed"], cache["v_packed"], cache["k_scale"],
                                    cache["v_scale"], nrep, g)
        dev = [cache[n].to(gpu) for n in ("k_packed", "v_packed", "k_scale", "v_scale")]
        qd = _rows(q, qform, gpu, torch.bfloat16)
        qd.copy_(q)
        # fp32 results at the attention's bar; 16-bit ones add their rounding (2^-9, 2^-12 relative)
        for dtype, rtol in ((torch.float32, 2e-3), (torch.bfloat16, 8e-3), (torch.float16, 3e-3)):
            out = _rows(q, oform, gpu, dtype)
            _abi.int4_prefill_attention(qd, *dev, out, nrep, g)
            assert_close_rel(out.float().cpu(), ref, rtol=rtol, what=f"{b}x{hkv}x{nrep} {dtype}")
