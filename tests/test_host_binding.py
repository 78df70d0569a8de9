"""The host binding: it declines what is not a plain call, and a plain call gives the ctypes path's
results and errors."""
import pytest
import torch

from layer_quant_amd import _abi
from hybrid_quant import int4_8b_attention as ia
from hybrid_quant import mamba_state_8b_kernel as ms


def test_binding_is_built_and_declines_tensors_off_the_gpu():
    host = _abi.host_binding()
    assert host, "the host binding is not built"
    t = torch.zeros(2, 2, 2, 16)
    assert host.int4_pack_kv(t, t, t, t, 32) is None
    assert host.int4_pack_kv_pair(*[t] * 7, 32) is None
    assert host.int4_decode_attention(*[t] * 5, None, t, 1, 1, 32, _abi._workspace.on_index) is None
    assert host.int4_decode_attention_pack(*[t] * 7, None, t, 1, 1, 32, _abi._workspace.on_index) is None
    assert host.int4_prefill_attention(*[t] * 6, 1, 32) is None
    assert host.mx_encode(*[t] * 4, None, 8, 0, 0, 0) is None
    assert host.mx_state_update(*[None] * 14, 8, True, 0, 0, 0) is None
    assert host.selective_state_update(*[t] * 10, True) is None
    with pytest.raises(TypeError):
        host.mx_encode(t)
    with pytest.raises(RuntimeError, match="GPU only"):
        _abi.mx_encode(t, t, t, t, 8)


def _both(monkeypatch, call):
    """call() through the binding and through ctypes: (result or exception) of each."""
    got = []
    for host in (_abi.host_binding(), False):
        monkeypatch.setattr(_abi, "_host", host)
        if not host:
            monkeypatch.setattr(_abi, "host_binding", lambda: False)
        try:
            got.append(call())
        except Exception as e:  # noqa: BLE001
            got.append((type(e), str(e)))
    monkeypatch.undo()
    return got


@pytest.mark.gpu
@pytest.mark.parametrize("seq_len", [1, 40, 4000, 5000])
def test_attention_matches_ctypes(gpu, monkeypatch, seq_len):
    gen = torch.Generator(device=gpu).manual_seed(seq_len)
    holder = type("Cache", (), {})()
    cache = ia._ensure_layer_cache(holder, 0, 2, 8, 4096, 128, 64, gpu)
    k = torch.randn(2, 8, 4096, 128, device=gpu, generator=gen).to(torch.bfloat16)
    ia._pack_kv_into_cache(cache, k, k.flip(2), torch.arange(4096, device=gpu), 64)
    q = torch.randn(2, 32, 1, 128, device=gpu, generator=gen).to(torch.bfloat16)
    mask = torch.ones(2, seq_len, device=gpu)
    a, b = _both(monkeypatch, lambda: ia._decode_attention(q, cache, seq_len, 4, 64, mask))
    assert (a == b) if isinstance(a, tuple) else torch.equal(a, b)
    assert isinstance(a, tuple) == (seq_len > 4096)
    a, b = _both(monkeypatch, lambda: ia._pack_and_decode_attention(
        q, k[:, :, :1], k[:, :, 1:2], cache, seq_len, 4, 64))
    assert (a == b) if isinstance(a, tuple) else torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("device_step", [False, True])
@pytest.mark.parametrize("heads", [16, 15])  # 15: not divisible by the 8 groups
def test_update_matches_ctypes(gpu, monkeypatch, device_step, heads):
    gen = torch.Generator(device=gpu).manual_seed(heads)
    h0 = torch.randn(2, heads, 8, 128, device=gpu, generator=gen)
    x = torch.randn(2, heads, 8, device=gpu, generator=gen).to(torch.bfloat16)
    dt = torch.rand(2, heads, 1, device=gpu, generator=gen).expand(2, heads, 8)
    A = -torch.rand(heads, 1, 1, device=gpu, generator=gen).expand(heads, 8, 128)
    B = torch.randn(2, 8, 128, device=gpu, generator=gen).to(torch.bfloat16)

    def call():
        cache = ms.allocate_state_kernel_cache(h0, format_bits=4)
        cache.step = 3
        if device_step:
            ms.enable_device_step(cache)
        y = ms.mx_state_selective_update(cache, x, dt, A, B, B.flip(0))
        return y, cache.q_state, cache.shared_exp, cache.micro_exp

    a, b = _both(monkeypatch, call)
    if heads == 15:
        assert a == b and a[0] is _abi.LQError
    else:
        assert all(torch.equal(s, t) for s, t in zip(a, b))
