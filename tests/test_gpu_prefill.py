"""The prefill kernels against 64-bit references: RoPE with its KV outputs and
causal GQA attention, at tile edges, ragged lengths and every shape of head
group, and LlamaPrefill's KV outputs in the layouts a caller may pass."""
import math

import pytest
import torch

from rngd_pd_amd import _lib
from rngd_pd_amd.kernels.handoff import stream_handle

pytestmark = pytest.mark.gpu
D = 128
BF16 = torch.bfloat16


def _rope64(t, inv):
    ang = torch.arange(t.shape[0], dtype=torch.float32)[:, None] * inv[None]
    c, s = ang.double().cos()[:, None], ang.double().sin()[:, None]
    a, b = t[..., :D // 2], t[..., D // 2:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _attend64(q, k, v):
    T, NH, NKV = q.shape[0], q.shape[1], k.shape[1]
    out = torch.empty_like(q)
    mask = torch.full((T, T), float("-inf"), dtype=torch.float64).triu(1)
    for h in range(NH):
        kv = h // (NH // NKV)
        p = torch.softmax(q[:, h] @ k[:, kv].t() / math.sqrt(D) + mask, -1)
        out[:, h] = p @ v[:, kv]
    return out


def _run(cuda, T, NH, NKV, qkv, inv, pad):
    """Rotated qkv, k, v [T, NKV, D] and the attention; k and v rows ``pad`` wider."""
    lib, st = _lib.lib(), stream_handle()
    table = torch.empty((T, D // 2, 2), dtype=torch.float32, device=cuda)
    n = lib.pdk_prefill_kv_tile_elems(T, NKV)
    nan = lambda *s: torch.full(s, float("nan"), dtype=BF16, device=cuda)   # noqa: E731
    kt, vt, out = nan(n), nan(n), nan(T + 2, NH * D)
    k, v = nan(T + 2, NKV * D + pad), nan(T + 2, NKV * D + pad)
    x = qkv.to(cuda)
    _lib.call("pdk_rope_table", inv.data_ptr(), T, D // 2, table.data_ptr(), st)
    _lib.call("pdk_prefill_rope_kv", x.data_ptr(), table.data_ptr(), T, NH, NKV, D, k.data_ptr(),
              k.stride(0), v.data_ptr(), v.stride(0), kt.data_ptr(), vt.data_ptr(), st)
    _lib.call("pdk_prefill_attn", x.data_ptr(), x.stride(0), kt.data_ptr(), vt.data_ptr(), T, NH,
              NKV, D, 1.0 / math.sqrt(D), out.data_ptr(), st)
    torch.cuda.synchronize()
    for t in (out, k, v):
        assert t[T:].isnan().all(), "rows past T written"
    if pad:
        assert k[:, NKV * D:].isnan().all() and v[:, NKV * D:].isnan().all()
    rows = lambda t: t[:T, :NKV * D].reshape(T, NKV, D).cpu()   # noqa: E731
    return x.cpu(), rows(k), rows(v), out[:T].reshape(T, NH, D).cpu()


@pytest.mark.parametrize("T,NH,NKV,pad", [
    (1, 4, 1, 0), (2, 8, 8, 8), (31, 8, 2, 0), (32, 8, 2, 0), (33, 8, 2, 128), (64, 6, 2, 0),
    (65, 3, 1, 0), (96, 16, 2, 0), (127, 4, 4, 0), (129, 32, 8, 0), (257, 5, 1, 0),
    (515, 8, 2, 0)])
def test_rope_and_attention(cuda, T, NH, NKV, pad):
    print(f"prefill attention T={T} NH={NH} NKV={NKV}", flush=True)
    g = torch.Generator().manual_seed(T * 100 + NH)
    qkv = torch.randn((T, (NH + 2 * NKV) * D), generator=g)
    qkv[:, :NH * D] *= 3                     # scores wide enough that the maximum moves
    qkv = qkv.to(BF16)
    inv = (1.0 / 10000.0 ** (torch.arange(D // 2, dtype=torch.float64) / (D // 2))).float()
    x, k, v, out = _run(cuda, T, NH, NKV, qkv, inv.to(cuda), pad)
    ref = qkv.double().view(T, NH + 2 * NKV, D)
    assert torch.equal(v, qkv.view(T, -1, D)[:, NH + NKV:])
    rot = _rope64(ref[:, :NH + NKV], inv)
    got = torch.cat([x[:, :NH * D].view(T, NH, D), k], 1).double()
    # One bf16 rounding (8 significant bits: at most 2^-8 of the value) of an
    # fp32 rotation whose products are at most the largest element.
    bound = rot.abs() * 2 ** -8 + ref[:, :NH + NKV].abs().max() * 2 ** -20
    worst = float(((got - rot).abs() / bound).max())
    assert worst <= 1, worst
    # The attention of what it was given (the rounded q and k): one bf16
    # rounding of fp32 sums. The scores carry 2^-21 of their largest terms'
    # sum (|q||k| / sqrt(D), up to about 2^6 here), so the weights 2^-15.
    q64, k64, v64 = got[:, :NH], got[:, NH:], v.double()
    want = _attend64(q64, k64, v64)
    err = (out.double() - want).abs()
    worst = float((err / (want.abs() * 2 ** -8 + v64.abs().max() * 2 ** -15)).max())
    assert worst <= 1, worst


def test_forward_fills_any_kv_out(cuda):
    """kv_out as the halves of one [L, 2, T, H, D] tensor, as wider rows, and
    in layouts and types the kernels do not write (filled by copies)."""
    from rngd_pd_amd.engines.llama_decode import LlamaConfig, LlamaWeights
    from rngd_pd_amd.engines.llama_prefill import LlamaPrefill
    cfg = LlamaConfig(hidden=256, n_heads=4, n_kv_heads=2, head_dim=128, inter=256, vocab=300,
                      n_layers=2)
    pre = LlamaPrefill(LlamaWeights.random(cfg, seed=1, device=cuda))
    T = 45
    tokens = list(range(T))
    first, k, v = pre.forward(tokens)
    e = lambda *s, **kw: torch.empty(s, device=cuda, **{"dtype": BF16, **kw})   # noqa: E731
    both, wide = e(2, 2, T, 2, D), e(2, T, 2, 2, D)
    flat = e(2 * 2 * T * 2 * D + 1)[1:].view(2, 2, T, 2, D)          # 2-byte aligned
    seen = []
    for out in ((both[:, 0], both[:, 1]), (wide[:, :, 0], wide[:, :, 1]),
                (flat[:, 0], flat[:, 1]),
                (e(2, T, D, 2).transpose(2, 3), e(2, 2, T, D).transpose(1, 2)),
                (e(2, T, 2, D, dtype=torch.float32), e(2, T, 2, D, dtype=torch.float32))):
        got = pre.forward(tokens, kv_out=out, on_layer=lambda li, a, b: seen.append((li, a, b)))
        torch.cuda.synchronize()
        assert got[0] == first and got[1] is out[0] and got[2] is out[1]
        assert torch.equal(out[0].to(BF16), k) and torch.equal(out[1].to(BF16), v)
        for li, a, b in seen[-2:]:
            assert a.data_ptr() == out[0][li].data_ptr() and b.data_ptr() == out[1][li].data_ptr()
    assert [s[0] for s in seen] == [0, 1] * 5
    with pytest.raises(RuntimeError):
        pre.forward(tokens, kv_out=(e(2, T + 1, 2, D), e(2, T + 1, 2, D)))


def test_other_head_dims(cuda):
    """head_dim 64 takes the torch path and gives the same KV for the same rows."""
    from rngd_pd_amd.engines.llama_decode import LlamaConfig, LlamaWeights
    from rngd_pd_amd.engines.llama_prefill import LlamaPrefill
    cfg = LlamaConfig(hidden=256, n_heads=4, n_kv_heads=2, head_dim=64, inter=260, vocab=300,
                      n_layers=2)
    pre = LlamaPrefill(LlamaWeights.random(cfg, seed=2, device=cuda))
    tokens = list(range(40))
    _, k, v = pre.forward(tokens)
    _, k2, v2 = pre.forward(tokens[:20])
    torch.cuda.synchronize()
    # The library may split a product of another height differently: bf16 noise.
    for a, b in ((k[:, :20], k2), (v[:, :20], v2)):
        assert (a.float() - b.float()).norm() <= 1e-2 * b.float().norm()
