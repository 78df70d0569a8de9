"""The MFMA prefill's row accesses and key groups: every form of the query and output rows (16-byte
accesses or element accesses) with one and with two key groups, at the edges of the 32-position
blocks and at the first tiles of the key loop, against the float64 oracle."""
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


def _key_groups(b, hkv, nrep, L, cus=256):
    """The key groups that the call takes (two_key_groups in int4_prefill.hip, 256 CUs)."""
    tiles = -(-L // 32)
    workgroups = b * hkv * -(-tiles * nrep // 4)
    two = tiles >= 3 if workgroups <= cus else workgroups <= min(2 * cus, 24 * tiles)
    return 2 if two else 1


# (b, hkv, nrep): the small grids take two key groups from three tiles on, the large ones one
GRIDS = {"two groups": [(1, 2, 4), (2, 1, 1), (1, 1, 8), (1, 2, 2)],
         "one group": [(16, 8, 4), (32, 16, 1)]}


@pytest.mark.parametrize("grid", list(GRIDS))
@pytest.mark.parametrize("L", [1, 31, 32, 33, 64, 65, 129, 200])
@pytest.mark.parametrize("qform,oform", [("contiguous", "contiguous"), ("transposed", "odd rows"),
                                         ("odd base", "transposed"), ("columns", "columns")])
def test_prefill_forms(gpu, diag, grid, L, qform, oform):
    diag.set("LQ_PREFILL_REQUIRE_MFMA")
    if grid == "one group":
        L += 100 if L < 129 else 0
    for i, (b, hkv, nrep) in enumerate(GRIDS[grid]):
        assert _key_groups(b, hkv, nrep, L) == (2 if grid == "two groups" and L > 64 else 1)
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


# 1 x 2 x 4: one workgroup per tile and unit; 33 x 8 x 1: 264 workgroups up to four tiles
@pytest.mark.parametrize("groups,b,hkv,nrep", [(2, 1, 2, 4), (1, 33, 8, 1)])
@pytest.mark.parametrize("L", [32, 64, 65, 96, 97, 128, 160, 161])
@pytest.mark.parametrize("span", [0, 13])
def test_first_tiles(gpu, diag, groups, b, hkv, nrep, L, span):
    """One to six key tiles: the ends of the prefetch (the next tile, the one after it, none) with one
    and with two key groups; with a span, V scales down to 2^-13 of their largest."""
    diag.set("LQ_PREFILL_REQUIRE_MFMA")
    groups = groups if L > 64 else 1
    assert _key_groups(b, hkv, nrep, L) == groups
    g = (32, 64, 128)[L % 3]
    gen = torch.Generator().manual_seed(L + span)
    cache = oik.allocate_cache(b, hkv, L + 3, 128, g)
    k, v = (torch.randn(b, hkv, L, 128, generator=gen) for _ in range(2))
    v *= torch.exp2(-torch.rand(b, hkv, L, 1, generator=gen) * span)
    oik.pack_kv_into_cache(cache, k.to(torch.bfloat16), v.to(torch.bfloat16), torch.arange(L), g)
    q = (torch.randn(b, hkv * nrep, L, 128, generator=gen) * 2).to(torch.bfloat16)
    ref = oik.prefill_attention(q, cache["k_packed"], cache["v_packed"], cache["k_scale"],
                                cache["v_scale"], nrep, g)
    dev = [cache[n].to(gpu) for n in ("k_packed", "v_packed", "k_scale", "v_scale")]
    out = torch.full(q.shape, float("nan"), device=gpu)
    _abi.int4_prefill_attention(q.to(gpu), *dev, out, nrep, g)
    assert_close_rel(out.cpu(), ref, what=f"L={L} groups={groups} span={span}")
