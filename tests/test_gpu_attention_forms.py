"""The decode attention's row loads and split merge: query and token rows of every form (loaded to
LDS directly where they are contiguous and 4-byte aligned, element by element otherwise) give the
same bits, and the merge is right at the edges of its split counts and head sizes."""
import pytest
import torch

from helpers import assert_close_rel
from layer_quant_amd import _abi
from oracle import int4_kv as oik

pytestmark = pytest.mark.gpu
NAMES = ("k_packed", "v_packed", "k_scale", "v_scale")


def _rows(x, form, device):
    """x [B, H, 1, D] on the device with rows of the form."""
    b, h, _, d = x.shape
    if form == "contiguous":
        return x.to(device)
    if form == "padded":       # rows apart by an even number of elements
        t = torch.zeros(b, h, 1, d + 6, dtype=x.dtype, device=device)[..., :d]
    elif form == "odd rows":
        t = torch.zeros(b, h, 1, d + 1, dtype=x.dtype, device=device)[..., :d]
    elif form == "odd base":
        t = torch.zeros(b * h * d + 8, dtype=x.dtype, device=device)[1:1 + b * h * d].view(x.shape)
    elif form == "heads last":  # [B, 1, H, D] of a projection
        t = torch.zeros(b, 1, h, d, dtype=x.dtype, device=device).transpose(1, 2)
    elif form == "one row":    # every head the same row (stride 0)
        return x[:, :1].to(device).expand(b, h, 1, d)
    else:                      # head_dim not contiguous
        t = torch.zeros(b, h, 1, d, 2, dtype=x.dtype, device=device)[..., 0]
    return t.copy_(x)


@pytest.mark.parametrize("form", ["padded", "odd rows", "odd base", "heads last", "columns", "one row"])
@pytest.mark.parametrize("nrep,g", [(1, 32), (2, 64), (4, 32), (8, 64), (16, 128)])
@pytest.mark.parametrize("s", [1, 33, 700])
def test_row_forms_give_the_same_bits(gpu, diag, form, nrep, g, s):
    diag.set("LQ_ATTN_REQUIRE_FAST")
    b, hkv, d = 2, 2, 128
    gen = torch.Generator().manual_seed(100 * nrep + s)
    cache = oik.allocate_cache(b, hkv, s + 2, d, g)
    k, v = (torch.randn(b, hkv, s, d, generator=gen).to(torch.bfloat16) for _ in range(2))
    oik.pack_kv_into_cache(cache, k, v, torch.arange(s), g)
    q = torch.randn(b, hkv * nrep, 1, d, generator=gen).to(torch.bfloat16)
    kn, vn = (torch.randn(b, hkv, 1, d, generator=gen).to(torch.bfloat16) for _ in range(2))
    if form == "one row":
        q, kn, vn = (t[:, :1].expand(t.shape).contiguous() for t in (q, kn, vn))

    def run(f):
        dev = [cache[n].to(gpu) for n in NAMES]
        out = torch.empty(b, hkv * nrep, d, device=gpu)
        rows = [_rows(t, f, gpu) for t in (q, kn, vn)]
        _abi.int4_decode_attention_pack(*rows, *dev, None, out, s, nrep, g)
        again = torch.empty_like(out)
        _abi.int4_decode_attention(rows[0], *dev, None, again, s, nrep, g)
        assert torch.equal(out, again)
        return [out, *dev]

    got, want = run(form), run("contiguous")
    assert all(torch.equal(a, b_) for a, b_ in zip(got, want))
    oik.pack_into(cache["k_packed"], cache["k_scale"], kn, torch.tensor([s - 1]), g)
    oik.pack_into(cache["v_packed"], cache["v_scale"], vn, torch.tensor([s - 1]), g)
    ref = oik.decode_attention(q, *(cache[n] for n in NAMES), s, nrep, g)
    assert_close_rel(got[0].cpu(), ref, what=form)


@pytest.mark.parametrize("d", [32, 64, 96, 128, 256, 260, 512])
@pytest.mark.parametrize("splits", [1, 2, 4, 5, 9, 16, 17, 33, 64, 65, 80])
def test_merge_split_counts(gpu, diag, d, splits):
    """The generic kernel's plan gives S / 64 splits here: every merge form and its edges."""
    diag.set("LQ_ATTN_FORCE_GENERIC")
    b, hkv, nrep, s = 1, 2, 2, 64 * splits - 5
    g = 4 if d == 260 else 32
    gen = torch.Generator().manual_seed(d + splits)
    cache = oik.allocate_cache(b, hkv, s, d, g)
    k, v = (torch.randn(b, hkv, s, d, generator=gen).to(torch.bfloat16) for _ in range(2))
    oik.pack_kv_into_cache(cache, k, v, torch.arange(s), g)
    q = torch.randn(b, hkv * nrep, 1, d, generator=gen)
    mask = torch.zeros(b, 1, 1, s)
    mask[..., : s // 3] = float("-inf")  # whole splits without a key
    for m in (None, mask):
        out = torch.full((b, hkv * nrep, d), float("nan"), device=gpu)
        _abi.int4_decode_attention(q.to(gpu), *(cache[n].to(gpu) for n in NAMES),
                                   None if m is None else m.to(gpu), out, s, nrep, g)
        ref = oik.decode_attention(q, *(cache[n] for n in NAMES), s, nrep, g, m)
        assert_close_rel(out.cpu(), ref, what=f"d={d} splits={splits}")


def test_all_keys_masked_is_nan_over_splits(gpu):
    b, hkv, nrep, s, d, g = 1, 8, 4, 2000, 128, 64
    cache = oik.allocate_cache(b, hkv, s, d, g)
    x = torch.randn(b, hkv, s, d).to(torch.bfloat16)
    oik.pack_kv_into_cache(cache, x, x, torch.arange(s), g)
    q = torch.randn(b, hkv * nrep, 1, d).to(torch.bfloat16).to(gpu)
    mask = torch.full((b, 1, 1, s), float("-inf"), device=gpu)
    out = torch.zeros(b, hkv * nrep, d, device=gpu)
    _abi.int4_decode_attention(q, *(cache[n].to(gpu) for n in NAMES), mask, out, s, nrep, g)
    assert torch.isnan(out).all()
