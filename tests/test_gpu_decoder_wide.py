"""LlamaDecoder beyond 16 streams at Llama-3.1-8B widths, where gate|up, the
lm_head and the down projection take the wide kernels and the down projection's
workspace is one for all layers, batch sizes and captured graphs: steps against
the oracle, and every stream bit for bit as in a step of its own."""
import numpy as np
import pytest
import torch

from tests.test_gpu_decode_step import _prefilled, _run_steps

pytestmark = pytest.mark.gpu


def _config():
    from rngd_pd_amd.engines.llama_decode import LlamaConfig
    return LlamaConfig(vocab=12300, n_layers=2)      # 193 groups of 64 columns, the last ragged


def test_steps_match_the_oracle(cuda):
    ctx = [1 + (37 * i) % 300 for i in range(50)]
    print("8B widths: 2 layers, B=50", flush=True)
    dec = _run_steps(cuda, _config(), ctx, steps=2, seed=17)
    assert dec.down_ws is not None


def test_a_stream_does_not_depend_on_its_batch(cuda):
    """Graphs of 50, 33, 17 and 16 streams of one decoder, replayed in turn with
    eager steps between: each stream's residual, logits and token are those of its
    step alone, and the workspace's counters end at zero."""
    from rngd_pd_amd.engines.llama_decode import LlamaDecoder, LlamaWeights
    cfg, rng = _config(), np.random.default_rng(23)
    ctx = [1 + (53 * i) % 700 for i in range(50)]
    w = LlamaWeights.random(cfg, seed=23, device=cuda)
    cache, tables, _, _ = _prefilled(cuda, cfg, ctx, 1, rng)
    dec = LlamaDecoder(w, cache, max_batch=50)
    assert dec.down_ws is not None
    tok = torch.from_numpy(rng.integers(0, cfg.vocab, 50)).to(cuda)
    ctx_d = torch.tensor(ctx, dtype=torch.int32, device=cuda)
    cap = tables.shape[1] * 16
    bits = lambda t: t.contiguous().view(torch.int16)   # noqa: E731
    dec.reserve(cap)
    alone = []
    for b in range(50):
        dec.step(tok[b:b + 1], ctx_d[b:b + 1], tables[b:b + 1], cap)
        alone.append((bits(dec.x[0]).clone(), bits(dec.logits[0]).clone(), int(dec.tokens[0])))
    graphs = {B: dec.capture(tok[:B], ctx_d[:B], tables[:B], cap) for B in (50, 33, 17, 16)}
    for B in (50, 17, 16, 33, 50, 17):
        print(f"replay B={B}", flush=True)
        dec.x_buf.zero_()
        dec.logits.zero_()
        dec.tokens.fill_(-1)
        torch.cuda.synchronize()
        graphs[B].replay()
        torch.cuda.synchronize()
        x, logits, tokens = bits(dec.x), bits(dec.logits), dec.tokens.tolist()
        for b in range(B):
            assert torch.equal(x[b], alone[b][0]), (B, b)
            assert torch.equal(logits[b], alone[b][1]) and tokens[b] == alone[b][2], (B, b)
        dec.step(tok[3:40], ctx_d[3:40], tables[3:40], cap)       # eager between replays
        torch.cuda.synchronize()
        assert torch.equal(bits(dec.x)[0], alone[3][0])
        assert int(dec.down_ws[:4096].abs().sum()) == 0
