"""Performance cases: the calls that a program serving a patched Nemotron-H model makes on the GPU.

Geometry throughout is the 8B model's: attention with 32 query and 8 KV heads of 128 dims over an
INT4 KV cache (group 32, 64 or 128), Mamba2 state of 128 heads x 64 x 128 with 8 B/C groups.

Kinds of case
  attn      one attention layer's decode step: pack the new token, attend over the packed cache;
            with `mask` the batch is left-padded and the call gets the 2-D keep-mask
  layer     the same through the patched model layer (projections, cache, output projection)
  prefill   causal attention of a prompt over its packed cache
  pack      a prompt's K and V quantised into the cache
  mx        one Mamba2 layer's decode step on an MX8 / MX4 state (stochastic writeback)
  ssm       the same on the plain bf16 state (layers that keep it, and the drift baseline)
  encode    a layer's state quantised when its MX cache is registered after the prompt
"""
from __future__ import annotations

import math

import torch
import torch.nn as nn

from layer_quant_amd import int4_8b_attention as ia
from layer_quant_amd import mamba_state_8b_kernel as ms

DEV = "cuda"
HQ, HKV, D = 32, 8, 128
NREP = HQ // HKV
HIDDEN = HQ * D
NH, P, N, NG = 128, 64, 128, 8


def listed():
    return [
        # one user's chat, short context, the driver's default group: latency and launches
        dict(name="attn_b1_ctx1000_g64", kind="attn", batch=1, ctx=1000, group=64, mask=False),
        # a padded batch of mid-length conversations
        dict(name="attn_mask_b8_ctx4001_g32", kind="attn", batch=8, ctx=4001, group=32, mask=True),
        # the benchmark's serving load: a full batch at long context
        dict(name="attn_b64_ctx16384_g32", kind="attn", batch=64, ctx=16384, group=32, mask=False),
        # a whole attention layer at the batch and context the reference publishes
        dict(name="layer_b8_ctx2072_g64", kind="layer", batch=8, ctx=2072, group=64),
        # short prompts of two users, and one long document
        dict(name="prefill_b2_l777_g64", kind="prefill", batch=2, length=777, group=64),
        dict(name="prefill_b1_l8192_g32", kind="prefill", batch=1, length=8192, group=32),
        # filling the cache from a long prompt
        dict(name="pack_b1_l16384_g32", kind="pack", batch=1, length=16384, group=32),
        # Mamba2 decode: the benchmark's full batch, the reference's batch, a few users
        dict(name="mx4_b64", kind="mx", batch=64, bits=4, layout="reference"),
        dict(name="mx8_b8", kind="mx", batch=8, bits=8, layout="reference"),
        dict(name="mx4_compact_b3", kind="mx", batch=3, bits=4, layout="compact"),
        # a layer kept in bf16
        dict(name="ssm_bf16_b16", kind="ssm", batch=16),
        # registration of the states after a prompt
        dict(name="encode_mx8_b8", kind="encode", batch=8, bits=8, layout="reference"),
    ]


def _log_int(rng, lo, hi):
    """A whole number between lo and hi, spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["attn", "attn", "attn", "layer", "prefill", "prefill", "pack", "mx", "mx",
                       "ssm", "encode"])
    group = rng.choice([32, 64, 128])
    batch = _log_int(rng, 1, 64)
    if kind == "attn":
        return dict(kind=kind, batch=batch, ctx=_log_int(rng, 64, 16384), group=group,
                    mask=rng.random() < 0.3)
    if kind == "layer":
        return dict(kind=kind, batch=_log_int(rng, 1, 32), ctx=_log_int(rng, 64, 8192), group=group)
    if kind == "prefill":
        batch = _log_int(rng, 1, 4)
        return dict(kind=kind, batch=batch, group=group,
                    length=_log_int(rng, 100, int(8192 / math.sqrt(batch))))
    if kind == "pack":
        batch = _log_int(rng, 1, 8)
        return dict(kind=kind, batch=batch, length=_log_int(rng, 64, 16384 // batch), group=group)
    if kind == "ssm":
        return dict(kind=kind, batch=batch)
    return dict(kind=kind, batch=batch, bits=rng.choice([4, 8]),
                layout=rng.choice(["reference", "reference", "compact"]))


# ---------------------------------------------------------------------------------------------
# inputs: plain torch, from the seed alone (prepare() and exact() both start from them)
# ---------------------------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(gen, *shape):
    return torch.randn(*shape, device=DEV, generator=gen)


def _kv(gen, *shape):
    """Keys or values with a few loud channels, as projections give them."""
    x = _randn(gen, *shape)
    x[..., ::37] *= 6.0
    return x.to(torch.bfloat16)


def _quantize(x, group):
    """INT4 levels and scales of x [..., D]: packed uint8 [..., D/2], fp32 [..., D/group]."""
    g = x.float().unflatten(-1, (x.shape[-1] // group, group))
    scale = (g.abs().amax(-1, keepdim=True) / 7.0).clamp_min(1e-8)
    level = (g / scale).round_().clamp_(-8, 7).flatten(-2).to(torch.int8).view(torch.uint8) & 15
    return level[..., 0::2] | (level[..., 1::2] << 4), scale.squeeze(-1)


def _dequantize(packed, scale, group):
    """float64 values of packed rows."""
    level = torch.stack((packed & 15, packed >> 4), -1).flatten(-2).to(torch.int16)
    level = torch.where(level > 7, level - 16, level).double()
    return (level.unflatten(-1, (-1, group)) * scale.double()[..., None]).flatten(-2)


def _filled_cache(gen, batch, rows, capacity, group):
    """k_packed, v_packed, k_scale, v_scale of `capacity` rows with `rows` tokens in them."""
    out = [torch.zeros(batch, HKV, capacity, w, device=DEV, dtype=t)
           for w, t in ((D // 2, torch.uint8), (D // 2, torch.uint8),
                        (D // group, torch.float32), (D // group, torch.float32))]
    per = max(1, (1 << 27) // (HKV * max(rows, 1) * D))
    for b in range(0, batch, per):
        n = min(per, batch - b)
        for i in range(2):
            packed, scale = _quantize(_kv(gen, n, HKV, rows, D), group)
            out[i][b:b + n, :, :rows] = packed
            out[2 + i][b:b + n, :, :rows] = scale
    return out


def _keep_mask(batch, ctx):
    """Left-padded batch: row b starts after its own number of padding tokens."""
    pad = (torch.arange(batch, device=DEV) * 977) % max(1, ctx // 2)
    return (torch.arange(ctx, device=DEV)[None, :] >= pad[:, None]).long()


def _mx_quantize(h, bits):
    """MX levels of a float state [..., N]: int8 [..., N], uint8 [..., N/16], uint8 [..., N/2]."""
    most = 63.0 if bits == 8 else 7.0
    blocks = h.float().unflatten(-1, (-1, 8, 2))
    pair = blocks.abs().amax(-1)
    exp = torch.ceil(torch.log2((pair.amax(-1) / (2 * most)).clamp_min(1e-30))).clamp(-126, 127)
    base = torch.exp2(exp)[..., None]
    micro = (pair > most * base).float()
    level = torch.round((blocks.abs() / (base * torch.exp2(micro))[..., None]).clamp_max(most))
    q = torch.where(blocks < 0, -level, level).flatten(-3).to(torch.int8)
    return q, (exp + 127).to(torch.uint8), micro.flatten(-2).to(torch.uint8)


def _mamba_inputs(gen, batch):
    """x, dt, A, B, C, D, dt_bias of one decode step, expanded as the model passes them."""
    bf = torch.bfloat16
    return dict(
        x=_randn(gen, batch, NH, P).to(bf),
        dt=_randn(gen, batch, NH).to(bf)[:, :, None].expand(batch, NH, P),
        A=(-torch.exp(torch.rand(NH, device=DEV, generator=gen) * 2))[:, None, None].expand(NH, P, N),
        B=_randn(gen, batch, NG, N).to(bf),
        C=_randn(gen, batch, NG, N).to(bf),
        D=_randn(gen, NH)[:, None].expand(NH, P),
        dt_bias=(_randn(gen, NH) * 0.1)[:, None].expand(NH, P))


def _state(gen, batch):
    return _randn(gen, batch, NH, P, N) * 0.5


def _compact(q, m, bits):
    """The compact layout's mantissas and micro-exponent bits."""
    if bits == 4:
        u = q.view(torch.uint8) & 15
        q = u[..., 0::2] | (u[..., 1::2] << 4)
    m = (m.unflatten(-1, (-1, 8)).int() << torch.arange(8, device=DEV, dtype=torch.int32)).sum(-1)
    return q.contiguous(), m.to(torch.uint8)


# ---------------------------------------------------------------------------------------------
# the model layer of the `layer` cases
# ---------------------------------------------------------------------------------------------
def repeat_kv(x, n_rep):
    b, h, s, d = x.shape
    return x[:, :, None].expand(b, h, n_rep, s, d).reshape(b, h * n_rep, s, d)


class _Attention(nn.Module):
    """The attention mixer's weights and attributes that the patched forward uses."""

    def __init__(self, seed):
        super().__init__()
        gen = _gen(seed)
        self.layer_idx = 0
        self.num_heads, self.num_key_value_heads, self.num_key_value_groups = HQ, HKV, NREP
        self.head_dim, self.hidden_size, self.attention_dropout = D, HIDDEN, 0.0
        for name, width in (("q_proj", HIDDEN), ("k_proj", HKV * D), ("v_proj", HKV * D),
                            ("o_proj", HIDDEN)):
            proj = nn.Linear(HIDDEN, width, bias=False, device="meta")
            w = (_randn(gen, width, HIDDEN) / math.sqrt(HIDDEN)).to(torch.bfloat16)
            proj.weight = nn.Parameter(w, requires_grad=False)
            setattr(self, name, proj)


class _Block(nn.Module):
    block_type = "attention"

    def __init__(self, seed):
        super().__init__()
        self.mixer = _Attention(seed)


class _Model(nn.Module):
    def __init__(self, seed):
        super().__init__()
        self.backbone = nn.Module()
        self.backbone.layers = nn.ModuleList([_Block(seed)])


class _PastKeyValue:
    """Stands for the model's cache object, on which the packed layer caches live."""


# ---------------------------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------------------------
def _attn_inputs(case, seed):
    gen, b, s, g = _gen(seed), case["batch"], case["ctx"], case["group"]
    cap = max(16, 1 << math.ceil(math.log2(s)))
    cache = _filled_cache(gen, b, s - 1, cap, g)
    if case["kind"] == "layer":
        return cache, _randn(gen, b, 1, HIDDEN).to(torch.bfloat16)
    q = _randn(gen, b, HQ, 1, D).to(torch.bfloat16)
    return cache, q, _kv(gen, b, HKV, 1, D), _kv(gen, b, HKV, 1, D)


def _prompt_cache(case, seed):
    gen, b, n, g = _gen(seed), case["batch"], case["length"], case["group"]
    cap = max(16, 1 << math.ceil(math.log2(n)))
    if case["kind"] == "prefill":
        cache = _filled_cache(gen, b, n, cap, g)
        return cache, _randn(gen, b, HQ, n, D).to(torch.bfloat16)
    return _kv(gen, b, HKV, n, D), _kv(gen, b, HKV, n, D), cap


def prepare(case, seed):
    kind = case["kind"]
    if kind == "attn":
        cache, q, k, v = _attn_inputs(case, seed)
        mask = _keep_mask(case["batch"], case["ctx"]) if case["mask"] else None
        cache = ia.Int4KVLayerCache(*cache, length=case["ctx"] - 1)
        return dict(case=case, cache=cache, q=q, k=k, v=v, mask=mask)
    if kind == "layer":
        cache, hidden = _attn_inputs(case, seed)
        model = _Model(seed)
        ia.patch_nemotron_h_attention_int4_kv(model, group_size=case["group"])
        past = _PastKeyValue()
        ia._cache_dict(past)[0] = ia.Int4KVLayerCache(*cache, length=case["ctx"] - 1)
        position = torch.tensor([case["ctx"] - 1], device=DEV)
        return dict(case=case, layer=model.backbone.layers[0].mixer, past=past, hidden=hidden,
                    position=position)
    if kind == "prefill":
        cache, q = _prompt_cache(case, seed)
        return dict(case=case, cache=ia.Int4KVLayerCache(*cache, length=case["length"]), q=q)
    if kind == "pack":
        k, v, cap = _prompt_cache(case, seed)
        shape = (case["batch"], HKV, cap)
        cache = ia.Int4KVLayerCache(
            torch.zeros(*shape, D // 2, device=DEV, dtype=torch.uint8),
            torch.zeros(*shape, D // 2, device=DEV, dtype=torch.uint8),
            torch.zeros(*shape, D // case["group"], device=DEV),
            torch.zeros(*shape, D // case["group"], device=DEV))
        positions = torch.arange(case["length"], device=DEV)
        return dict(case=case, cache=cache, k=k, v=v, positions=positions)
    gen = _gen(seed)
    state = _state(gen, case["batch"])
    if kind == "encode":
        return dict(case=case, state=state.to(torch.bfloat16))
    inputs = _mamba_inputs(gen, case["batch"])
    if kind == "ssm":
        return dict(case=case, state=state.to(torch.bfloat16), inputs=inputs)
    q, e, m = _mx_quantize(state, case["bits"])
    if case["layout"] == "compact":
        q, m = _compact(q, m, case["bits"])
    cache = ms.MambaStateKernelCache(q_state=q, shared_exp=e, micro_exp=m,
                                     format_bits=case["bits"], layout=case["layout"])
    return dict(case=case, cache=cache, inputs=inputs)


def _tensors(cache):
    return [cache.k_packed, cache.v_packed, cache.k_scale, cache.v_scale]


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "attn":
        cache = state["cache"]
        out = ia._pack_and_decode_attention(state["q"], state["k"], state["v"], cache, case["ctx"],
                                            NREP, case["group"], attention_mask=state["mask"])
        return [out, *_tensors(cache)]
    if kind == "layer":
        past = state["past"]
        out, _, past = state["layer"].forward(state["hidden"], past_key_value=past, use_cache=True,
                                              cache_position=state["position"])
        return [out, *_tensors(ia._cache_dict(past)[0])]
    if kind == "prefill":
        return [ia._prefill_attention(state["q"], state["cache"], NREP, case["group"])]
    if kind == "pack":
        ia._pack_kv_into_cache(state["cache"], state["k"], state["v"], state["positions"],
                               case["group"])
        return [*_tensors(state["cache"]), state["cache"].length]
    if kind == "encode":
        cache = ms.allocate_state_kernel_cache(state["state"], format_bits=case["bits"],
                                               layout=case["layout"])
        return [cache.q_state, cache.shared_exp, cache.micro_exp]
    if kind == "ssm":
        y = ms.selective_state_update(state["state"], dt_softplus=True, **state["inputs"])
        return [y, state["state"]]
    cache = state["cache"]
    y = ms.mx_state_selective_update(cache, dt_softplus=True, **state["inputs"])
    return [y, cache.q_state, cache.shared_exp, cache.micro_exp]


# ---------------------------------------------------------------------------------------------
# what a pass cannot do without, how far results may be apart, and the answer in 64 bits
# ---------------------------------------------------------------------------------------------
def work(case):
    kind, b = case["kind"], case["batch"]
    if kind in ("attn", "layer"):
        row = D + 2 * 4 * (D // case["group"])  # K and V bytes of one token and head
        kv = b * HKV * case["ctx"] * row
        flops = 4.0 * b * HQ * case["ctx"] * D
        new = b * HKV * D * 2 * 2
        if kind == "attn":
            mask = 8 * b * case["ctx"] if case["mask"] else 0
            return dict(bytes=kv + mask + new + 2 * b * HQ * D * 2, flops=flops)
        weights = 2 * HIDDEN * (2 * HIDDEN + 2 * HKV * D)
        return dict(bytes=kv + weights + 2 * b * HIDDEN * 2, flops=flops + weights * b)
    if kind == "prefill":
        n = case["length"]
        row = D + 2 * 4 * (D // case["group"])
        return dict(bytes=b * n * (HKV * row + 2 * HQ * D * 2),
                    flops=4.0 * D * b * HQ * n * (n + 1) / 2)
    if kind == "pack":
        tokens = 2 * b * HKV * case["length"]
        return dict(bytes=tokens * (2 * D + D // 2 + 4 * (D // case["group"])), flops=0)
    values = b * NH * P * N
    if kind == "encode":
        return dict(bytes=int(values * (2 + _mx_bytes(case))), flops=0)
    small = b * NH * P * 4 + b * (2 * NG * N * 2 + NH * 2) + 3 * NH * 4
    if kind == "ssm":
        return dict(bytes=values * 4 + small, flops=5 * values)
    return dict(bytes=int(2 * values * _mx_bytes(case)) + small, flops=5 * values)


def _mx_bytes(case):
    """State bytes per value."""
    if case["layout"] == "reference":
        return 1 + 1 / 16 + 1 / 2
    return (1 if case["bits"] == 8 else 0.5) + 1 / 16 + 1 / 16


def tolerance(case):
    kind = case["kind"]
    if kind in ("pack", "encode"):
        return "exact"
    if kind == "layer":  # bf16 projections around the attention
        return {"rel": 1e-2, "max": 0.1, "differ": 0.0}
    if kind == "mx":  # levels on the edge of a rounding step may fall either way
        return {"rel": 7e-3, "max": 0.03, "differ": 2e-4}
    return {"rel": 7e-3, "max": 0.03, "differ": 0.0}  # bf16 results


def _exact_attention(q, cache, group, keep=None, causal=False):
    """softmax(q k^T / sqrt(D)) v in 64 bits: q [B, HQ, T, D] over the cache's rows."""
    kp, vp, ks, vs = cache
    out = torch.empty(q.shape, device=DEV, dtype=torch.float64)
    for b in range(q.shape[0]):
        for h in range(HKV):
            k = _dequantize(kp[b, h], ks[b, h], group)
            v = _dequantize(vp[b, h], vs[b, h], group)
            for i in range(NREP * h, NREP * (h + 1)):
                s = (q[b, i].double() @ k.t().contiguous()) / math.sqrt(D)
                if keep is not None:
                    s.masked_fill_(keep[b][None, :] == 0, -math.inf)
                if causal:
                    s.masked_fill_(torch.ones_like(s, dtype=torch.bool).triu_(1), -math.inf)
                out[b, i] = torch.softmax(s, -1) @ v
    return out


def _with_token(cache, k, v, row, group):
    """The cache's first row + 1 rows, with the token k, v packed into the last."""
    for i, x in enumerate((k, v)):
        packed, scale = _quantize(x, group)
        cache[i][:, :, row] = packed[:, :, 0]
        cache[2 + i][:, :, row] = scale[:, :, 0]
    return [t[:, :, :row + 1] for t in cache]


def _exact_update(h, inputs):
    """y and the new state of one step in 64 bits."""
    f = {name: t.double() for name, t in inputs.items() if name != "A"}
    dt = torch.nn.functional.softplus(f["dt"] + f["dt_bias"])[:, :, 0]
    decay = torch.exp(inputs["A"][:, 0, 0].double() * dt)[:, :, None, None]
    rep = NH // NG
    drive = f["B"].repeat_interleave(rep, 1)[:, :, None, :] * (dt[:, :, None] * f["x"])[..., None]
    h = h.double() * decay + drive
    y = (h * f["C"].repeat_interleave(rep, 1)[:, :, None, :]).sum(-1) + f["x"] * f["D"]
    return y, h


def exact(case, seed):
    kind = case["kind"]
    if kind in ("pack", "encode"):
        return None  # bytes
    if kind == "prefill":
        cache, q = _prompt_cache(case, seed)
        rows = [t[:, :, :case["length"]] for t in cache]
        return [_exact_attention(q, rows, case["group"], causal=True)]
    if kind == "attn":
        cache, q, k, v = _attn_inputs(case, seed)
        rows = _with_token(cache, k, v, case["ctx"] - 1, case["group"])
        keep = _keep_mask(case["batch"], case["ctx"]) if case["mask"] else None
        out = _exact_attention(q, rows, case["group"], keep)
        return [out[:, :, 0], None, None, cache[2], cache[3]]
    if kind == "layer":
        cache, hidden = _attn_inputs(case, seed)
        m, b = _Attention(seed), case["batch"]
        x = hidden[:, 0].double()
        q, k, v = ((x @ p.weight.double().t().contiguous()).view(b, -1, 1, D)
                   for p in (m.q_proj, m.k_proj, m.v_proj))
        rows = _with_token(cache, k, v, case["ctx"] - 1, case["group"])
        out = _exact_attention(q, rows, case["group"]).reshape(b, 1, HIDDEN)
        return [out @ m.o_proj.weight.double().t().contiguous(), None, None, None, None]
    gen = _gen(seed)
    state = _state(gen, case["batch"])
    inputs = _mamba_inputs(gen, case["batch"])
    if kind == "ssm":
        return list(_exact_update(state.to(torch.bfloat16), inputs))
    q, e, m = _mx_quantize(state, case["bits"])
    scale = torch.exp2(e.double().repeat_interleave(16, -1) - 127 + m.double().repeat_interleave(2, -1))
    return [_exact_update(q.double() * scale, inputs)[0], None, None, None]
