"""The decode attention's split merge at the end of fp32's range: infinite partials beside finite
ones."""
import pytest
import torch

from helpers import assert_close_rel
from layer_quant_amd import _abi
from oracle import int4_kv as oik

pytestmark = pytest.mark.gpu
NAMES = ("k_packed", "v_packed", "k_scale", "v_scale")


def _run(gpu, q, k, v, g):
    """The GPU's and the oracle's attention of q [1, Hq, 1, D] over the packed k, v [1, Hkv, S, D]."""
    _, hkv, s, d = k.shape
    nrep = q.shape[1] // hkv
    cache = oik.allocate_cache(1, hkv, s, d, g)
    oik.pack_kv_into_cache(cache, k, v, torch.arange(s), g)
    out = torch.full((1, hkv * nrep, d), float("nan"), device=gpu)
    _abi.int4_decode_attention(q.to(gpu), *(cache[n].to(gpu) for n in NAMES), None, out, s, nrep, g)
    return out.cpu(), oik.decode_attention(q, *(cache[n] for n in NAMES), s, nrep, g)


@pytest.mark.parametrize("where", ["first", "last"])
@pytest.mark.parametrize("splits", [2, 5, 9, 17, 33, 64, 65])
def test_infinite_partial_stays_infinite(gpu, diag, splits, where):
    """Equal scores; the first 32 dims of one split's values overflow its fp32 sum. 64 keys per split
    (the generic kernel's plan): every split count of the merge kernels, with and without a repeated
    last split."""
    diag.set("LQ_ATTN_FORCE_GENERIC")
    s, d = 64 * splits - 5, 64
    gen = torch.Generator().manual_seed(splits)
    k, v = torch.zeros(1, 2, s, d), torch.randn(1, 2, s, d, generator=gen)
    rows = slice(0, 64) if where == "first" else slice(64 * (splits - 1), s)
    v[:, :, rows, :32] = 3.0e38
    out, ref = _run(gpu, torch.randn(1, 4, 1, d, generator=gen), k, v, 32)
    assert torch.isposinf(out[..., :32]).all()
    assert_close_rel(out[..., 32:], ref[..., 32:], what=f"splits={splits}")
