"""Decode attention under an int64 keep-mask read by the kernel: the same bytes as with its additive
bias, with and without the new token, on the MFMA and the generic path."""

import pytest
import torch

from layer_quant_amd import _abi
from layer_quant_amd import int4_8b_attention as ia
from test_abi_cpu import _fake


def test_keep_rejects_bad_arguments():
    f = _abi.lib().lq_int4_decode_attention_keep
    kp, ks = _fake((2, 8, 64, 64), torch.uint8), _fake((2, 8, 64, 4), torch.float32)
    q, out = _fake((2, 32, 1, 128), torch.bfloat16), _fake((2, 32, 128), torch.bfloat16)
    kn, keep = _fake((2, 8, 1, 128), torch.bfloat16), _fake((2, 10), torch.int64)
    tail = (out, 10, 4, 32, None, 0, None)
    for bad in (None, _fake((3, 10), torch.int64), _fake((2, 10), torch.int32),
                _fake((2, 1, 1, 10), torch.int64)):
        assert f(q, kn, kn, kp, kp, ks, ks, bad, *tail) == _abi.LQ_ERR_INVALID_ARG
    assert f(q, kn, None, kp, kp, ks, ks, keep, *tail) == _abi.LQ_ERR_INVALID_ARG
    # the entries with a bias go on refusing a keep-mask
    g = _abi.lib().lq_int4_decode_attention
    assert g(q, kp, kp, ks, ks, keep, *tail) == _abi.LQ_ERR_INVALID_ARG


def test_only_dense_int64_rows_are_read_as_they_are():
    cpu = torch.device("cpu")
    keep = torch.ones(2, 9, dtype=torch.int64)
    assert torch.equal(ia._keep_rows(keep, 2, 7, cpu), keep[:, 2:])
    assert ia._keep_rows(keep[:1].expand(2, 9), 2, 9, cpu) is not None
    for other in (None, keep.bool(), keep.int(), keep[:1], keep.t().contiguous().t(),
                  keep[:, :1].expand(2, 9), keep[:, None, None], keep.to("meta")):
        assert ia._keep_rows(other, 2, 9, cpu) is None
    assert ia._keep_rows(keep, 2, 10, cpu) is None


@pytest.mark.gpu
@pytest.mark.parametrize("generic", [False, True])
@pytest.mark.parametrize("nrep,g", [(1, 128), (4, 32), (4, 64), (8, 64)])
@pytest.mark.parametrize("s", [1, 31, 32, 33, 63, 64, 65, 97, 1000, 4129])
def test_keep_equals_its_bias(gpu, diag, generic, nrep, g, s):
    if generic:
        diag.set("LQ_ATTN_FORCE_GENERIC")
    b, hkv, d = 3, 2, 128
    gen = torch.Generator().manual_seed(s + nrep)

    def bf16(*shape):
        return torch.randn(*shape, generator=gen).to(torch.bfloat16).to(gpu)

    q, kn, vn, k, v = bf16(b, 2 * nrep, 1, d), bf16(b, hkv, 1, d), bf16(b, hkv, 1, d), \
        bf16(b, hkv, s, d), bf16(b, hkv, s, d)
    packed = [torch.zeros(b, hkv, s + 3, d // 2, dtype=torch.uint8, device=gpu) for _ in range(2)]
    scales = [torch.zeros(b, hkv, s + 3, d // g, device=gpu) for _ in range(2)]
    _abi.int4_pack_kv_pair(k, v, *packed, *scales, torch.arange(s, device=gpu), g)
    # every nonzero value keeps its key, also one whose low or high word is zero; the second row
    # masks whole tiles, the third everything but the newest key; rows start at odd columns
    keep = torch.tensor([0, 1, -1, 1 << 32, 2])[torch.randint(0, 5, (b, s + 3), generator=gen)]
    keep[:, -1] = 1
    keep[1, : 3 + s // 2] = 0
    keep[2, :-1] = 0
    keep = keep.to(gpu)
    rows = ia._keep_rows(keep, b, s, gpu)
    bias = torch.zeros(b, 1, 1, s, device=gpu).masked_fill((rows == 0)[:, None, None], -torch.inf)

    def run(call, token, mask):
        out = torch.full((b, 2 * nrep, d), torch.nan, device=gpu)
        dev = [t.clone() for t in (*packed, *scales)]
        call(q, *token, *dev, mask, out, s, nrep, g)
        return [out, *dev]

    for token, plain in (((kn, vn), _abi.int4_decode_attention_pack),
                         ((), _abi.int4_decode_attention)):
        want = run(plain, token, bias)
        got = run(_abi.int4_decode_attention_keep, token or (None, None), rows)
        assert not torch.isnan(got[0]).any()
        assert all(torch.equal(x, y) for x, y in zip(got, want))
        # a mask that ends before the last key masks the rest
        short = rows[:, : s // 2]
        if s > 1:
            want = run(plain, token, bias[..., : s // 2].contiguous())
            got = run(_abi.int4_decode_attention_keep, token or (None, None), short)
            assert all(torch.equal(x.nan_to_num(7.0), y.nan_to_num(7.0)) for x, y in zip(got, want))
