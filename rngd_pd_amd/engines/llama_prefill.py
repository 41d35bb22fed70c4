"""Llama prefill for the producer side of the handoff: prompt -> per-layer KV + first token.

Stands in for FullPrefillEngine.prefill_stream (engines/prefill_full.py:337-388)
on MI355X: the prompt's K/V per layer (after RoPE, bf16, token-major
[T, Hkv, D] as the connector's device save takes them) and the greedy next
token of the last position (the reference's "next", serving/cluster.py:
330-343). Each layer's K/V is handed to ``on_layer`` as soon as the layer is
done, so saves overlap the layers that follow (the reference emits layer
groups as it goes).

Up to 256 tokens the GEMMs are pdk_prefill_gemm's (K split over workgroups, fp32
partial sums that the next kernel adds up), the O and down projections' up to
512; a longer prompt is compute-bound on tiles enough for every CU and its GEMMs
are the library's (hipBLASLt through torch). At head_dim 128, one launch per line
of a layer, the short prompt's on the right:

  h = rmsnorm(x + down)                pdk_rmsnorm          pdk_prefill_rmsnorm_partials
  qkv = h . Wqkv^T                     library              pdk_prefill_gemm
  RoPE; K/V rows; attention's operands pdk_prefill_rope_kv  pdk_prefill_rope_kv_partials
  ao = causal GQA attention            pdk_prefill_attn (fp32 weights)
  o = ao . Wo^T                        library              pdk_prefill_gemm
  h = rmsnorm(x + o)                   pdk_rmsnorm          pdk_prefill_rmsnorm_partials
  gu = h . Wgu^T                       library              pdk_prefill_gemm_swiglu, with
  act = silu(g) * u                    pdk_swiglu             this line
  down = act . Wd^T                    library              pdk_prefill_gemm

Other head dims take RoPE and attention as fp32 torch operations on contiguous
operands. Activations are bf16 at tensor boundaries, as in the decode step. It
takes the decode step's LlamaWeights ([out, in] layout), so a producer and a
consumer built from one seed hold the same model.
"""
import math

import torch

from .. import _lib
from ..kernels.handoff import stream_handle

BF16 = torch.bfloat16


def _rows(t, shape, device):
    """The token stride of a layer's K or V rows ([T, Hkv, D] bf16, [Hkv, D]
    contiguous, 16-byte aligned) as pdk_prefill_rope_kv writes them, or None
    for any other tensor (filled by a copy instead)."""
    if t.dtype != BF16 or t.device != device or tuple(t.shape) != shape \
            or t.data_ptr() % 16 or t.stride(2) != 1 or t.stride(1) != shape[2]:
        return None
    ld = t.stride(0) if shape[0] > 1 else shape[1] * shape[2]
    return ld if ld >= shape[1] * shape[2] and ld % 8 == 0 else None


class _Partials:
    """A projection as ``splits`` fp32 partial sums [splits, T, N], to be added by
    the kernel that reads it."""

    def __init__(self, buf, splits, T, N):
        self.buf, self.splits, self.T, self.N = buf, splits, T, N


class _Projections:
    """The projections of one forward over T tokens. Those pdk_prefill_gemm takes
    write their partial sums to one workspace: each is read by the launch after
    it, before the next one writes."""

    def __init__(self, cfg, T, device):
        lib, H = _lib.lib(), cfg.hidden
        self.T, self.device, self.M = T, device, cfg.inter
        self.splits = {(N, K): lib.pdk_prefill_gemm_splits(T, K, N)
                       for N, K in ((cfg.qkv_dim, H), (H, cfg.n_heads * cfg.head_dim),
                                    (H, cfg.inter))}
        self.fused = bool(lib.pdk_prefill_gemm_swiglu_takes(T, H, cfg.inter))
        n = max(s * T * N for (N, _), s in self.splits.items())
        self.buf = torch.empty(n, dtype=torch.float32, device=device) if n else None

    def direct(self, w):
        """Whether a kernel can read this weight where it lies."""
        return w.dtype == BF16 and w.device == self.device and w.is_contiguous() \
            and w.data_ptr() % 16 == 0

    def linear(self, x, w, partials=True):
        """x . w^T: _Partials where the kernel takes the shape (and the caller
        takes partials), else bf16."""
        splits = self.splits.get(tuple(w.shape), 0) if partials else 0
        if not splits or not self.direct(w):
            return torch.nn.functional.linear(x, w)
        N, K = w.shape
        _lib.call("pdk_prefill_gemm", x.data_ptr(), w.data_ptr(), self.T, K, N,
                  self.buf.data_ptr(), stream_handle())
        return _Partials(self.buf, splits, self.T, N)

    def swiglu(self, x, w):
        """silu(x . wg^T) * (x . wu^T) in one launch, or None."""
        if not self.fused or tuple(w.shape) != (2 * self.M, x.shape[1]) or not self.direct(w):
            return None
        act = torch.empty((self.T, self.M), dtype=BF16, device=self.device)
        _lib.call("pdk_prefill_gemm_swiglu", x.data_ptr(), w.data_ptr(), self.T, x.shape[1],
                  self.M, act.data_ptr(), stream_handle())
        return act


class LlamaPrefill:
    def __init__(self, weights, max_tokens=4096):
        self.w, self.cfg = weights, weights.cfg
        self.device = weights.embed.device
        self.max_tokens = max_tokens
        cfg = self.cfg
        self.inv = cfg.inv_freq().to(self.device)
        self.scale = 1.0 / math.sqrt(cfg.head_dim)

    def _rmsnorm(self, x, weight, out, add=None, row=0):
        """out = rmsnorm(x + add) * weight over the rows of x from ``row``; with
        ``add``, x takes the sum."""
        if isinstance(add, _Partials):
            _lib.call("pdk_prefill_rmsnorm_partials", x[row:].data_ptr(),
                      add.buf.data_ptr() + 4 * row * add.N, add.T * add.N, add.splits,
                      weight.data_ptr(), add.T - row, add.N, self.cfg.eps, out.data_ptr(),
                      stream_handle())
            return out
        if row:
            x, add = x[row:], None if add is None else add[row:]
        T, H = x.shape
        _lib.call("pdk_rmsnorm", x.data_ptr(), None if add is None else add.data_ptr(),
                  weight.data_ptr(), T, H, self.cfg.eps, out.data_ptr(), stream_handle())
        return out

    def _rope(self, t, cos, sin):
        """t [T, n, HD] bf16 -> rotate-half RoPE in fp32 -> bf16."""
        half = t.shape[-1] // 2
        f = t.float()
        a, b = f[..., :half], f[..., half:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1).to(BF16)

    def _kernel_attention(self, T):
        """The layer's RoPE, KV rows and attention by the HIP kernels: a
        function (qkv, k_l, v_l, before) -> ao [T, NH HD] bf16; ``before`` is
        called once k_l and v_l are written."""
        cfg, dev, st = self.cfg, self.device, stream_handle()
        NH, NKV, HD = cfg.n_heads, cfg.n_kv_heads, cfg.head_dim
        table = torch.empty((T, HD // 2, 2), dtype=torch.float32, device=dev)
        _lib.call("pdk_rope_table", self.inv.data_ptr(), T, HD // 2, table.data_ptr(), st)
        n = _lib.lib().pdk_prefill_kv_tile_elems(T, NKV)
        kt, vt = (torch.empty(n, dtype=BF16, device=dev) for _ in range(2))
        ao = torch.empty((T, NH * HD), dtype=BF16, device=dev)
        q_rows = None

        def attention(qkv, k_l, v_l, before):
            nonlocal q_rows
            rows = []
            for t in (k_l, v_l):
                ld = _rows(t, (T, NKV, HD), dev)
                own = t if ld else torch.empty((T, NKV, HD), dtype=BF16, device=dev)
                rows.append((own, ld or NKV * HD))
            (k, k_ld), (v, v_ld) = rows
            outs = (k.data_ptr(), k_ld, v.data_ptr(), v_ld, kt.data_ptr(), vt.data_ptr(),
                    stream_handle())
            if isinstance(qkv, _Partials):
                if q_rows is None:
                    q_rows = torch.empty((T, NH * HD), dtype=BF16, device=dev)
                _lib.call("pdk_prefill_rope_kv_partials", qkv.buf.data_ptr(), qkv.splits,
                          table.data_ptr(), T, NH, NKV, HD, q_rows.data_ptr(), *outs)
                qkv = q_rows
            else:
                _lib.call("pdk_prefill_rope_kv", qkv.data_ptr(), table.data_ptr(), T, NH, NKV, HD,
                          *outs)
            if k is not k_l:
                k_l.copy_(k)
            if v is not v_l:
                v_l.copy_(v)
            before()
            _lib.call("pdk_prefill_attn", qkv.data_ptr(), qkv.stride(0), kt.data_ptr(),
                      vt.data_ptr(), T, NH, NKV, HD, self.scale, ao.data_ptr(), stream_handle())
            return ao

        return attention

    def _torch_attention(self, T):
        """The same for head dims the kernels do not take, in fp32 torch."""
        cfg, dev = self.cfg, self.device
        NH, NKV, HD = cfg.n_heads, cfg.n_kv_heads, cfg.head_dim
        G = NH // NKV
        pos = torch.arange(T, device=dev, dtype=torch.float32)
        ang = pos[:, None] * self.inv[None, :]                     # fp32 angles, [T, HD/2]
        cos, sin = torch.cos(ang)[:, None, :], torch.sin(ang)[:, None, :]
        causal = torch.full((T, T), float("-inf"), device=dev).triu(1)

        def attention(qkv, k_l, v_l, before):
            q = self._rope(qkv[:, :NH * HD].view(T, NH, HD), cos, sin)
            k = self._rope(qkv[:, NH * HD:(NH + NKV) * HD].view(T, NKV, HD), cos, sin)
            v = qkv[:, (NH + NKV) * HD:].view(T, NKV, HD)
            k_l.copy_(k)
            v_l.copy_(v)
            before()
            # Causal GQA attention in fp32: query head h reads KV head h // G.
            qf = q.float().view(T, NKV, G, HD).permute(1, 2, 0, 3).reshape(NKV, G * T, HD)
            kt = k.float().permute(1, 2, 0).contiguous()               # [NKV, HD, T]
            vf = v.float().permute(1, 0, 2).contiguous()               # [NKV, T, HD]
            sc = torch.bmm(qf.contiguous(), kt).view(NKV, G, T, T) * self.scale + causal
            p = torch.softmax(sc, dim=-1).view(NKV, G * T, T)
            ao = torch.bmm(p, vf).view(NKV, G, T, HD).permute(2, 0, 1, 3).reshape(T, NH * HD)
            return ao.to(BF16)

        return attention

    def _swiglu(self, gu):
        T, M = gu.shape[0], self.cfg.inter
        if M % 8:
            return (torch.nn.functional.silu(gu[:, :M].float()) * gu[:, M:].float()).to(BF16)
        act = torch.empty((T, M), dtype=BF16, device=gu.device)
        _lib.call("pdk_swiglu", gu.data_ptr(), T, M, act.data_ptr(), stream_handle())
        return act

    def _greedy(self, last, lm_head, proj):
        """The token of the largest logit of last [1, H] (the first of equals). The
        head is one row of the short prompts' GEMM; the host takes the largest of
        the few keys that the partial sums reduce to."""
        N, K = lm_head.shape
        splits = _lib.lib().pdk_prefill_gemm_splits(1, K, N) if proj.direct(lm_head) else 0
        if not splits:
            return int(torch.argmax(torch.nn.functional.linear(last, lm_head)[0]).item())
        part = torch.empty(splits * N, dtype=torch.float32, device=self.device)
        keys = torch.empty(-(-N // 1024), dtype=torch.int64, device=self.device)
        st = stream_handle()
        _lib.call("pdk_prefill_gemm", last.data_ptr(), lm_head.data_ptr(), 1, K, N,
                  part.data_ptr(), st)
        _lib.call("pdk_prefill_argmax", part.data_ptr(), splits, N, keys.data_ptr(), st)
        return 0xffffffff - (max(keys.tolist()) & 0xffffffff)

    @torch.no_grad()
    def forward(self, tokens, on_layer=None, kv_out=None):
        """tokens: int sequence or int64 tensor [T] (T >= 1). Returns (first
        token, k, v) with k, v bf16 [L, T, Hkv, D] (kv_out may supply them).
        on_layer(li, k_l, v_l) is called after each layer on the current stream."""
        cfg, w, dev = self.cfg, self.w, self.device
        ids = torch.as_tensor(tokens, dtype=torch.int64, device=dev).reshape(-1)
        T = ids.numel()
        if not 1 <= T <= self.max_tokens:
            raise ValueError(f"prompt of {T} tokens outside [1, {self.max_tokens}]")
        L, H, NKV, HD = cfg.n_layers, cfg.hidden, cfg.n_kv_heads, cfg.head_dim
        if kv_out is None:
            k_all = torch.empty((L, T, NKV, HD), dtype=BF16, device=dev)
            v_all = torch.empty((L, T, NKV, HD), dtype=BF16, device=dev)
        else:
            k_all, v_all = kv_out
        fused = HD == 128
        attention = (self._kernel_attention if fused else self._torch_attention)(T)
        proj = _Projections(cfg, T, dev)
        x = w.embed.index_select(0, ids)                           # [T, H] bf16
        h = torch.empty_like(x)
        down = None                                                # not yet added to x
        for li in range(L):
            self._rmsnorm(x, w.norm1[li], h, add=down)
            k_l, v_l = k_all[li], v_all[li]
            emit = (lambda: None) if on_layer is None else (lambda: on_layer(li, k_l, v_l))
            ao = attention(proj.linear(h, w.wqkv[li], partials=fused), k_l, v_l, emit)
            self._rmsnorm(x, w.norm2[li], h, add=proj.linear(ao, w.wo[li]))
            act = proj.swiglu(h, w.wgu[li])
            if act is None:
                act = self._swiglu(torch.nn.functional.linear(h, w.wgu[li]))
            down = proj.linear(act, w.wd[li])
        last = torch.empty((1, H), dtype=BF16, device=dev)
        self._rmsnorm(x, w.norm_f, last, add=down, row=T - 1)
        return self._greedy(last, w.lm_head, proj), k_all, v_all
