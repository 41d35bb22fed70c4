"""pdk_decode_attn_append (the new token's cache write inside the attention
launch) against pdk_cache_append followed by pdk_decode_attn: outputs and
caches equal bit for bit, over every plan (V whole and in halves, query heads
split, context split), positions at block and span edges, contexts without a
token, past the table and in invalid blocks, and tables that share blocks."""
import numpy as np
import pytest
import torch

from tests._util import rand_bf16, to_dev

pytestmark = pytest.mark.gpu


def _bits(t):
    return t.contiguous().view(torch.int16)


@pytest.mark.parametrize("B,Hq,Hkv,ctx", [
    (1, 32, 8, [1]), (1, 32, 8, [129]), (1, 8, 8, [2049]), (2, 16, 1, [513, 32]),
    (4, 32, 8, [512, 33, 16, 17]), (6, 32, 8, [700, 5800, 2049, 1024, 31, 4097]),
    (16, 32, 8, [512 - 13 * i for i in range(16)]), (20, 32, 8, [300 + 17 * i for i in range(20)]),
    (33, 8, 8, [64 + 31 * i for i in range(33)]), (36, 8, 8, [1 + 3 * i for i in range(36)]), (40, 64, 8, [8 + 16 * i for i in range(40)])])
def test_append_equals_two_calls(cuda, B, Hq, Hkv, ctx):
    from rngd_pd_amd import kernels as K
    D, rng = 128, np.random.default_rng(B * 31 + Hq)
    mb = -(-max(ctx) // 16) + 1
    nb = sum(-(-c // 16) for c in ctx) + 3
    ids = rng.permutation(nb).astype(np.int32)
    tables, at = np.full((B, mb), -1, np.int32), 0
    for b, c in enumerate(ctx):
        n = -(-c // 16)
        tables[b, :n] = ids[at:at + n]
        at += n
    ctx = list(ctx)
    if B >= 4:                                   # no token; past the table; an invalid block
        ctx[1], ctx[2] = 0, mb * 16 + 5
        tables[3, (ctx[3] - 1) // 16] = nb + 7
    print(f"append B={B} Hq={Hq} Hkv={Hkv} ctx={ctx[:6]}", flush=True)
    q, kn, vn = (to_dev(rand_bf16(rng, (B, h, D))) for h in (Hq, Hkv, Hkv))
    ck, cv = to_dev(rand_bf16(rng, (nb, Hkv, 16, D))), to_dev(rand_bf16(rng, (nb, Hkv, D, 16)))
    tab = torch.from_numpy(tables).to(cuda)
    ctx_t = torch.tensor(ctx, dtype=torch.int32, device=cuda)
    max_ctx = min(max(ctx), mb * 16)
    ck2, cv2 = ck.clone(), cv.clone()
    K.cache_append(kn, vn, ck, cv, tab, ctx_t)
    want = K.decode_attention(q, ck, cv, tab, ctx_t, max_ctx, scale=0.088)
    wide = torch.zeros((B, Hkv, 2, D), dtype=torch.bfloat16, device=cuda)
    wide[:, :, 0] = kn
    out = torch.full_like(q, float("nan"))
    K.decode_attention_append(q, wide[:, :, 0], vn, ck2, cv2, tab, ctx_t, max_ctx, scale=0.088,
                              out=out)
    torch.cuda.synchronize()
    assert torch.equal(_bits(ck), _bits(ck2)) and torch.equal(_bits(cv), _bits(cv2))
    assert torch.equal(_bits(out), _bits(want))
    # 2-byte aligned rows take the two launches.
    odd = torch.zeros(B * Hkv * D + 1, dtype=torch.bfloat16, device=cuda)
    odd[1:] = vn.reshape(-1)
    got = K.decode_attention_append(q, kn, odd[1:].view(B, Hkv, D), ck2, cv2, tab, ctx_t, max_ctx,
                                    scale=0.088)
    torch.cuda.synchronize()
    assert torch.equal(_bits(got), _bits(want))


@pytest.mark.parametrize("Hq,Hkv,groups", [
    # (last context, rows) of each request: its rows stand at consecutive positions
    (32, 8, [(40, 4)]), (8, 8, [(18, 3), (33, 2), (5, 1)]), (16, 1, [(2050, 5)]),
    (32, 8, [(5000, 3), (700, 2), (20, 1)]), (32, 8, [(512 + 7 * i, 4) for i in range(4)]),
    (32, 8, [(1100 + i, 3) for i in range(7)]), (8, 8, [(150 + 33 * i, 4) for i in range(16)]),
    (16, 2, [(300 + 9 * i, 17) for i in range(3)]), (8, 2, [(64, 64)]),
    (8, 2, [(70, 65)])])                             # beyond a wavefront's lanes: two launches
def test_streams_that_share_blocks(cuda, Hq, Hkv, groups):
    """Rows of one request at consecutive positions in one call: each attends over
    the new tokens of those before it, bit for bit as in two calls."""
    from rngd_pd_amd import kernels as K
    D, rng = 128, np.random.default_rng(len(groups) * 100 + Hq)
    mb = -(-max(c for c, _ in groups) // 16) + 1
    nb = sum(-(-c // 16) for c, _ in groups) + 3
    ids, at, tables, ctx = rng.permutation(nb).astype(np.int32), 0, [], []
    for c, n in groups:
        row = np.full(mb, -1, np.int32)
        blocks = -(-c // 16)
        row[:blocks] = ids[at:at + blocks]
        row[blocks:] = row[blocks - 1]               # past the context: takes no part
        if c - n >= 16 and n > 3:                    # the written block, earlier as well (and
            row[0] = row[blocks - 1]                 # no row's own slot twice)
        at += blocks
        for i in range(n):
            tables.append(row)
            ctx.append(c - n + 1 + i)
    order = rng.permutation(len(ctx))
    tables, ctx = np.stack(tables)[order], [ctx[i] for i in order]
    B = len(ctx)
    print(f"shared blocks B={B} Hq={Hq} Hkv={Hkv} ctx={ctx[:8]}", flush=True)
    q, kn, vn = (to_dev(rand_bf16(rng, (B, h, D))) for h in (Hq, Hkv, Hkv))
    ck, cv = to_dev(rand_bf16(rng, (nb, Hkv, 16, D))), to_dev(rand_bf16(rng, (nb, Hkv, D, 16)))
    tab = torch.from_numpy(tables).to(cuda)
    ctx_t = torch.tensor(ctx, dtype=torch.int32, device=cuda)
    ck2, cv2 = ck.clone(), cv.clone()
    K.cache_append(kn, vn, ck, cv, tab, ctx_t)
    want = K.decode_attention(q, ck, cv, tab, ctx_t, max(ctx), scale=0.088)
    got = K.decode_attention_append(q, kn, vn, ck2, cv2, tab, ctx_t, max(ctx), scale=0.088)
    torch.cuda.synchronize()
    assert torch.equal(_bits(ck), _bits(ck2)) and torch.equal(_bits(cv), _bits(cv2))
    assert torch.equal(_bits(got), _bits(want))


@pytest.mark.parametrize("which", ["k", "v"])
def test_output_over_the_new_rows(cuda, which):
    from rngd_pd_amd import kernels as K
    B, H, D, rng = 5, 8, 128, np.random.default_rng(3)
    q, kn, vn = (to_dev(rand_bf16(rng, (B, H, D))) for _ in range(3))
    ck, cv = to_dev(rand_bf16(rng, (20, H, 16, D))), to_dev(rand_bf16(rng, (20, H, D, 16)))
    tab = torch.arange(20, dtype=torch.int32, device=cuda).view(B, 4)
    ctx = torch.tensor([64, 33, 16, 1, 50], dtype=torch.int32, device=cuda)
    ck2, cv2 = ck.clone(), cv.clone()
    want = K.decode_attention_append(q, kn, vn, ck, cv, tab, ctx, 64)
    out = kn if which == "k" else vn
    got = K.decode_attention_append(q, kn, vn, ck2, cv2, tab, ctx, 64, out=out)
    torch.cuda.synchronize()
    assert torch.equal(_bits(ck), _bits(ck2)) and torch.equal(_bits(cv), _bits(cv2))
    assert torch.equal(_bits(got), _bits(want))
