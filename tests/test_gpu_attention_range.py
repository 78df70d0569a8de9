"""The decode attention's merges at the ends of fp32's range: infinite partials beside finite ones,
and weights below the smallest normal number."""
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


@pytest.mark.parametrize("fast,s,cold", [(False, 64 * n - 5, 64) for n in (2, 9, 33, 65)]
                         + [(True, 128, 32), (True, 128 * 2, 128), (True, 128 * 20 - 7, 128)])
def test_subnormal_weight_of_large_values(gpu, diag, fast, s, cold):
    """The first `cold` keys score 127.5 below the others (in powers of two), and their values are
    2^126 times larger, so that their subnormal weight still makes a quarter of the result or more. They are
    one split's keys, or (fast, 128 keys) one wave's tile of 32."""
    diag.set("LQ_ATTN_REQUIRE_FAST" if fast else "LQ_ATTN_FORCE_GENERIC")
    gen = torch.Generator().manual_seed(s)
    q = torch.full((1, 4, 1, 128), 7.8125, dtype=torch.bfloat16)  # q . k = 1000 for k = 1
    k, v = torch.ones(1, 2, s, 128), torch.randn(1, 2, s, 128, generator=gen)
    k[:, :, :cold] = 0.0
    v[:, :, :cold] = v[:, :, :cold].abs() * 2.0 ** 118
    v[:, :, cold:] *= 2.0 ** -8
    out, ref = _run(gpu, q, k, v, 32)
    assert_close_rel(out, ref, what=f"fast={fast} S={s}")
