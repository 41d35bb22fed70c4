"""The decode step's GEMMs for 17 to 64 rows (wgemm_wide.hip) against the
row-major entry points, which run wgemm_kernel: the canonical order of the sum
over K makes them equal bit for bit, at the edges of the row tiles, with a last
column tile past N, and on both sides of the rules that choose the kernel. That
wgemm_kernel is right is test_gpu_decode_step.py's."""
import numpy as np
import pytest
import torch

from rngd_pd_amd import _lib
from tests._util import rand_bf16, to_dev
from tests.test_gpu_act_tiled import _eq, _tiled_in

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def _operands(cuda, B, K, rows):
    from rngd_pd_amd import kernels as K_
    rng = np.random.default_rng(B + K + rows)
    x = to_dev(rand_bf16(rng, (B, K)))
    g = torch.Generator(device=cuda).manual_seed(B + rows)
    w = (torch.randn((rows, K), generator=g, device=cuda) * 0.05).to(BF16)
    ssq = torch.from_numpy(rng.random((B, K // 16)).astype(np.float32) + 0.5).to(cuda)
    return x, K_.tile_weight(w), ssq


@pytest.mark.parametrize("B,K,M", [(17, 2048, 12288), (32, 4096, 12288), (33, 2048, 14336),
                                   (50, 4096, 14336), (64, 2048, 12288), (40, 1152, 12288),
                                   (64, 2048, 12160)])
def test_swiglu(cuda, B, K, M):
    from rngd_pd_amd import kernels as K_
    x, wt, ssq = _operands(cuda, B, K, 2 * M)
    print(f"wide swiglu B={B} K={K} M={M}", flush=True)
    ref = torch.empty((B, M), dtype=BF16, device=cuda)
    out = torch.full((K_.act_rows(B) * M,), float("nan"), dtype=BF16, device=cuda)
    for name, xin, y in (("tiled", x, ref), ("xt", _tiled_in(x), out)):
        _lib.call("pdk_linear_swiglu_rms_" + name, xin.data_ptr(), wt.data_ptr(), B, K, M,
                  ssq.data_ptr(), K // 16, 1e-5, y.data_ptr(), 0)
    torch.cuda.synchronize()
    assert _eq(K_.act_untile(out, B, M), ref)


@pytest.mark.parametrize("B,K,N", [(17, 2048, 12225), (33, 4096, 16032), (48, 2048, 12288),
                                   (64, 2048, 20001), (64, 1152, 12288), (20, 2048, 8016),
                                   (8, 2048, 8016), (16, 2048, 16032), (7, 2048, 6100),
                                   (33, 2048, 6160), (40, 4096, 8016), (48, 1152, 12225)])
def test_argmax(cuda, B, K, N):
    x, wt, ssq = _operands(cuda, B, K, N)
    print(f"wide argmax B={B} K={K} N={N}", flush=True)
    outs = []
    for name, xin in (("tiled", x), ("xt", _tiled_in(x)), ("xt", _tiled_in(x))):
        logits = torch.full((B + 1, N), float("nan"), dtype=BF16, device=cuda)
        keys = torch.zeros(B, dtype=torch.int64, device=cuda)
        tok = torch.full((B,), -1, dtype=torch.int32, device=cuda)
        _lib.call("pdk_linear_argmax_rms_" + name, xin.data_ptr(), wt.data_ptr(), B, K, N,
                  ssq.data_ptr(), K // 16, 1e-5, logits.data_ptr(), keys.data_ptr(),
                  tok.data_ptr(), 0)
        torch.cuda.synchronize()
        assert logits[B].isnan().all() and int(keys.abs().sum()) == 0
        outs.append((logits[:B], tok))
    for logits, tok in outs[1:]:
        assert _eq(logits, outs[0][0]) and torch.equal(tok, outs[0][1])


def test_one_workspace_for_several_shapes(cuda):
    """Calls of several widths in turn on one workspace, zeroed once."""
    from rngd_pd_amd import kernels as K_
    lib, K, shapes = _lib.lib(), 8192, [(64, 4096), (17, 4224), (33, 8192), (20, 4224)]
    ws = torch.zeros(max(lib.pdk_linear_ssq_ws_bytes(B, K, N) for B, N in shapes) // 4,
                     dtype=torch.int32, device=cuda)
    for B, N in shapes + shapes[::-1]:
        x, wt, _ = _operands(cuda, B, K, N)
        r = to_dev(rand_bf16(np.random.default_rng(N), (B, N), 4.0))
        print(f"shared workspace B={B} N={N}", flush=True)
        ref, ssq_ref = r.clone(), torch.zeros((B, N // 16), dtype=torch.float32, device=cuda)
        _lib.call("pdk_linear_ssq_tiled", x.data_ptr(), wt.data_ptr(), B, K, N, ref.data_ptr(),
                  ref.data_ptr(), ssq_ref.data_ptr(), 0)
        y = _tiled_in(r)
        ssq = torch.full((B, N // 16), float("nan"), dtype=torch.float32, device=cuda)
        _lib.call("pdk_linear_ssq_ws_xt", _tiled_in(x).data_ptr(), wt.data_ptr(), B, K, N,
                  y.data_ptr(), y.data_ptr(), ssq.data_ptr(), ws.data_ptr(), ws.numel() * 4, 0)
        torch.cuda.synchronize()
        assert _eq(K_.act_untile(y, B, N), ref) and torch.equal(ssq, ssq_ref), (B, N)


@pytest.mark.parametrize("B,K,N", [(17, 8192, 4096), (32, 14336, 4096), (33, 8192, 4224),
                                   (50, 14336, 4096), (64, 8192, 4096), (64, 4096, 4096),
                                   (16, 8192, 4096), (40, 8320, 4096)])
def test_ssq_with_workspace(cuda, B, K, N):
    from rngd_pd_amd import kernels as K_
    x, wt, _ = _operands(cuda, B, K, N)
    r = to_dev(rand_bf16(np.random.default_rng(B), (B, N), 4.0))
    lib = _lib.lib()
    need = lib.pdk_linear_ssq_ws_bytes(B, K, N)
    assert (need > 0) == (B > 16 and K % 2048 == 0 and K >= 8192)
    most = max(lib.pdk_linear_ssq_ws_bytes(64, K, N), 16)        # a workspace for 64 rows
    ws = torch.zeros(most // 4, dtype=torch.int32, device=cuda)
    print(f"wide ssq B={B} K={K} N={N} ws={need}", flush=True)
    ref, ssq_ref = r.clone(), torch.zeros((B, N // 16), dtype=torch.float32, device=cuda)
    _lib.call("pdk_linear_ssq_tiled", x.data_ptr(), wt.data_ptr(), B, K, N, ref.data_ptr(),
              ref.data_ptr(), ssq_ref.data_ptr(), 0)
    for call in range(3):                                        # the counters end at zero
        y = _tiled_in(r)
        ssq = torch.full((B, N // 16), float("nan"), dtype=torch.float32, device=cuda)
        _lib.call("pdk_linear_ssq_ws_xt", _tiled_in(x).data_ptr(), wt.data_ptr(), B, K, N,
                  y.data_ptr(), y.data_ptr(), ssq.data_ptr(), ws.data_ptr(), ws.numel() * 4, 0)
        torch.cuda.synchronize()
        assert _eq(K_.act_untile(y, B, N), ref) and torch.equal(ssq, ssq_ref), call
    if need:
        rc = lib.pdk_linear_ssq_ws_xt(x.data_ptr(), wt.data_ptr(), B, K, N, y.data_ptr(),
                                      y.data_ptr(), ssq.data_ptr(), ws.data_ptr(), need - 4, 0)
        assert rc == _lib.PDK_EINVAL and "workspace" in _lib.last_error()
