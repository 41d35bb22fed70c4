"""The short prompts' GEMMs against 64-bit products at the edges of their tiles and
splits, the kernels that add up their partial sums against the ones that take the
rounded projection, and LlamaPrefill on either side of every switch."""
import pytest
import torch

from rngd_pd_amd import _lib
from rngd_pd_amd.kernels.handoff import stream_handle

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def _rand(seed, *shape, std=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(shape, generator=g) * std).to(BF16)


@pytest.mark.parametrize("T,K,N", [
    (1, 256, 4), (1, 4096, 512), (15, 320, 132), (16, 1024, 128), (17, 256, 64), (31, 2112, 68),
    (32, 704, 60), (33, 256, 260), (64, 1088, 124), (65, 256, 128), (128, 960, 132),
    (129, 256, 252), (200, 4096, 256), (256, 320, 516), (257, 512, 4), (385, 1024, 260),
    (512, 14336, 256),
    # more than 32 tiles of 128 columns, or a K above 4096: the wider tiles
    (16, 256, 4100), (32, 320, 4100), (64, 4160, 100), (63, 256, 4228), (128, 4160, 132)])
def test_partials(cuda, T, K, N):
    s = _lib.lib().pdk_prefill_gemm_splits(T, K, N)
    print(f"prefill gemm T={T} K={K} N={N} splits={s}", flush=True)
    assert 1 <= s <= 8
    x, w = _rand(T, T, K), _rand(N, N, K, std=0.05)
    part = torch.full((s * T * N + 64,), float("nan"), dtype=torch.float32, device=cuda)
    xd, wd = x.to(cuda), w.to(cuda)
    _lib.call("pdk_prefill_gemm", xd.data_ptr(), wd.data_ptr(), T, K, N, part.data_ptr(),
              stream_handle())
    torch.cuda.synchronize()
    assert part[s * T * N:].isnan().all()
    got = part[:s * T * N].view(s, T, N).double().sum(0).cpu()
    # K fp32 additions of exact products: each rounds by 2^-24 of a sum that is at
    # most that of the absolute products.
    bound = K * 2.0 ** -24 * (x.abs().double() @ w.abs().double().t())
    assert ((got - x.double() @ w.double().t()).abs() <= bound).all()


@pytest.mark.parametrize("T,K,M", [(1, 256, 4), (16, 4096, 100), (17, 256, 32), (32, 320, 36),
                                   (40, 256, 64), (64, 1024, 68), (65, 256, 60), (128, 320, 132),
                                   (129, 256, 124), (256, 512, 132)])
def test_swiglu(cuda, T, K, M):
    print(f"prefill gemm swiglu T={T} K={K} M={M}", flush=True)
    assert _lib.lib().pdk_prefill_gemm_swiglu_takes(T, K, M) == 1
    x, w = _rand(T, T, K), _rand(M, 2 * M, K, std=0.1)
    y = torch.full((T * M + 64,), float("nan"), dtype=BF16, device=cuda)
    xd, wd = x.to(cuda), w.to(cuda)
    _lib.call("pdk_prefill_gemm_swiglu", xd.data_ptr(), wd.data_ptr(), T, K, M, y.data_ptr(),
              stream_handle())
    torch.cuda.synchronize()
    assert y[T * M:].isnan().all()
    got = y[:T * M].view(T, M).double().cpu()
    gu = x.double() @ w.double().t()
    e = K * 2.0 ** -24 * (x.abs().double() @ w.abs().double().t())
    g, u, eg, eu = gu[:, :M], gu[:, M:], e[:, :M], e[:, M:]
    a = torch.nn.functional.silu(g)
    # The two sums' errors (silu's slope is at most 1.1) and one bf16 rounding; the
    # fp32 exponential and division are within 2^-20 of the value.
    bound = 1.1 * eg * (u.abs() + eu) + a.abs() * eu + (a * u).abs() * (2.0 ** -8 + 2.0 ** -20)
    assert ((got - a * u).abs() <= bound + 1e-30).all()


@pytest.mark.parametrize("T,NH,NKV,splits", [(1, 4, 1, 5), (33, 3, 3, 1), (64, 8, 2, 8),
                                             (45, 2, 1, 4)])
def test_rope_from_partials(cuda, T, NH, NKV, splits):
    """The same bits as pdk_prefill_rope_kv on the rounded sum."""
    D, n = 128, (NH + 2 * NKV) * 128
    g = torch.Generator().manual_seed(T)
    part = torch.randn((splits, T, n), generator=g).to(cuda)
    total = torch.zeros((T, n), device=cuda)
    for p in part:
        total = total + p
    qkv, st = total.to(BF16), stream_handle()
    inv = (1.0 / 10000.0 ** (torch.arange(D // 2, dtype=torch.float64) / (D // 2))).float().to(cuda)
    table = torch.empty((T, D // 2, 2), dtype=torch.float32, device=cuda)
    _lib.call("pdk_rope_table", inv.data_ptr(), T, D // 2, table.data_ptr(), st)
    m = _lib.lib().pdk_prefill_kv_tile_elems(T, NKV)
    nan = lambda *s: torch.full(s, float("nan"), dtype=BF16, device=cuda)   # noqa: E731
    want = [nan(T, NKV, D), nan(T, NKV, D), nan(m), nan(m)]
    got = [nan(T, NKV, D), nan(T, NKV, D), nan(m), nan(m)]
    q = nan(T, NH * D)
    outs = lambda o: (o[0].data_ptr(), NKV * D, o[1].data_ptr(), NKV * D,   # noqa: E731
                      o[2].data_ptr(), o[3].data_ptr(), st)
    _lib.call("pdk_prefill_rope_kv_partials", part.data_ptr(), splits, table.data_ptr(), T, NH,
              NKV, D, q.data_ptr(), *outs(got))
    _lib.call("pdk_prefill_rope_kv", qkv.data_ptr(), table.data_ptr(), T, NH, NKV, D, *outs(want))
    torch.cuda.synchronize()
    assert torch.equal(q, qkv[:, :NH * D])
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("T,H,splits,first", [(1, 8, 1, 0), (5, 4096, 8, 0), (7, 8192, 5, 6),
                                              (3, 4104, 3, 1)])
def test_norm_from_partials(cuda, T, H, splits, first):
    x, w = _rand(1, T, H).to(cuda), (_rand(2, H) * 0.1 + 1).to(cuda)
    part = torch.randn((splits, T, H), generator=torch.Generator().manual_seed(3)).to(cuda)
    total = torch.zeros((T, H), device=cuda)
    for p in part:
        total = total + p
    want_x = (x.float() + total).to(BF16)
    got, out = x.clone(), torch.full((T - first, H), float("nan"), dtype=BF16, device=cuda)
    _lib.call("pdk_prefill_rmsnorm_partials", got[first:].data_ptr(),
              part[0, first:].data_ptr(), T * H, splits, w.data_ptr(), T - first, H, 1e-5,
              out.data_ptr(), stream_handle())
    torch.cuda.synchronize()
    assert torch.equal(got[first:], want_x[first:]) and torch.equal(got[:first], x[:first])
    x64 = want_x[first:].double()
    want = x64 * torch.rsqrt((x64 * x64).mean(-1, keepdim=True) + 1e-5) * w.double()
    # One bf16 rounding of an fp32 value (H additions: 2^-24 H / 2 of the scale).
    assert ((out.double() - want).abs() <= want.abs() * (2.0 ** -8 + H * 2.0 ** -25)).all()


@pytest.mark.parametrize("N,splits", [(4, 1), (1020, 3), (1028, 2), (16032, 2)])
def test_argmax_of_partials(cuda, N, splits):
    part = torch.randn((splits, N), generator=torch.Generator().manual_seed(N)).to(cuda)
    part[:, N // 2:] = part[:, :N - N // 2]                    # ties: the first counts
    total = torch.zeros(N, device=cuda)
    for p in part:
        total = total + p
    keys = torch.empty(-(-N // 1024), dtype=torch.int64, device=cuda)
    for case in ("plain", "inf", "nan"):
        if case != "plain":
            part[0, N - 1] = total[N - 1] = float(case)
        _lib.call("pdk_prefill_argmax", part.data_ptr(), splits, N, keys.data_ptr(),
                  stream_handle())
        got = 0xffffffff - (max(keys.tolist()) & 0xffffffff)
        assert got == int(torch.argmax(total.to(BF16).float().cpu())), case


@pytest.mark.parametrize("K,N", [(4096, 128256), (4096, 1028), (14336, 260), (256, 300),
                                 (4096, 1027), (320, 5000)])
def test_greedy_token(cuda, K, N):
    """The head's token where it is clear: one row of the head along the hidden
    state, anywhere in the vocabulary, and two equal ones (the first counts)."""
    from rngd_pd_amd.engines.llama_decode import LlamaConfig, LlamaWeights
    from rngd_pd_amd.engines.llama_prefill import LlamaPrefill, _Projections
    cfg = LlamaConfig(hidden=256, n_heads=2, n_kv_heads=1, head_dim=128, inter=256, vocab=64,
                      n_layers=1)
    pre = LlamaPrefill(LlamaWeights.random(cfg, seed=5, device=cuda))
    proj = _Projections(cfg, 1, pre.device)
    print(f"greedy K={K} N={N} splits={_lib.lib().pdk_prefill_gemm_splits(1, K, N)}", flush=True)
    g = torch.Generator(device=cuda).manual_seed(N)
    last = torch.randn((1, K), generator=g, device=cuda).to(BF16)
    head = (torch.randn((N, K), generator=g, device=cuda) * 0.02).to(BF16)
    # The other logits are N(0, 0.02 sqrt(K)); the row's own is 0.2 K, at least
    # 160 of their deviations.
    for row in sorted({0, 3, N // 2, min(1023, N - 2), min(1024, N - 1), N - 1}):
        kept = head[row].clone(), head[N - 1].clone()
        head[row] = last[0] * 0.2
        assert pre._greedy(last, head, proj) == row
        head[N - 1] = head[row]
        assert pre._greedy(last, head, proj) == row
        head[N - 1] = kept[1]
        head[row] = kept[0]


def test_forward_on_both_sides_of_the_switches(cuda):
    """A prompt's first tokens have the same KV whatever kernels its length
    takes, and a weight the kernels cannot read takes the library."""
    from rngd_pd_amd.engines.llama_decode import LlamaConfig, LlamaWeights
    from rngd_pd_amd.engines.llama_prefill import LlamaPrefill
    cfg = LlamaConfig(hidden=512, n_heads=4, n_kv_heads=2, head_dim=128, inter=768, vocab=300,
                      n_layers=3)
    w = LlamaWeights.random(cfg, seed=4, device=cuda)
    tokens = [(7 * i) % 300 for i in range(513)]
    _, k, v = LlamaPrefill(w).forward(tokens)                  # the library's GEMMs
    off = torch.empty(w.wo.numel() + 1, dtype=BF16, device=cuda)[1:].view_as(w.wo).copy_(w.wo)
    odd = LlamaWeights(cfg, w.norm1, w.wqkv.transpose(1, 2).contiguous().transpose(1, 2), off,
                       w.norm2, w.wgu, w.wd, w.embed, w.norm_f, w.lm_head)
    for weights, lengths in ((w, (1, 16, 17, 33, 65, 129, 256, 257, 512)), (odd, (40,))):
        for T in lengths:
            print(f"forward T={T}", flush=True)
            first, a, b = LlamaPrefill(weights).forward(tokens[:T])
            assert 0 <= first < 300
            for got, want in ((a, k[:, :T]), (b, v[:, :T])):
                # bf16 activations through three layers.
                assert (got.float() - want.float()).norm() <= 1e-2 * want.float().norm()
