"""Split plans of the GQA-4 decode at the edges of its one-chunk instance:
the most splits a fold holds (64), the most workgroups resident at once (512
on a 256-CU device), one token past a split, and ragged batches."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from .cqtest import assert_tight, build_gpu_cache, build_oracle
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,T,ragged", [
    (1, 8, 512, False), (1, 8, 513, False), (1, 8, 16385, False), (1, 2, 32768, False),
    (1, 2, 32769, False), (8, 8, 4096, True), (9, 8, 4096, True), (33, 2, 1100, True)])
def test_one_chunk_plan_edges(B, H, T, ragged):
    from chronoquant_mlx_amd.kernels import chronoquant_sdpa_cache_kernel, decode_status
    rng = np.random.default_rng(B * 131 + T)
    G, D, scale = 4, 128, 128 ** -0.5
    step = rng.standard_normal((B, H, T, D), dtype=np.float32) * 0.1
    k = np.cumsum(step, axis=2).astype(np.float16)
    v = np.cumsum(step[..., ::-1, :], axis=2).astype(np.float16)
    q = rng.standard_normal((B, G * H, D)).astype(np.float16)
    cache = build_gpu_cache(k, v, stride_k=32, stride_v=8)
    lens = rng.integers(0, T + 1, size=B) if ragged else np.full(B, T)
    if ragged:
        lens[:3] = [T, 1, 0]
    dl = torch.tensor(lens, dtype=torch.int32, device="cuda") if ragged else None
    qt = torch.from_numpy(q).cuda()
    outs = [chronoquant_sdpa_cache_kernel(qt, cache, scale, seq_lens=dl).cpu().numpy() for _ in range(2)]
    from chronoquant_mlx_amd import cache as cache_module
    stream = torch.cuda.current_stream()
    assert decode_status(cache_module._WORKSPACES[(stream.device.index, stream.cuda_stream)]) == 0
    assert np.array_equal(outs[0], outs[1])
    for b in sorted({0, 1, 2, B // 2, B - 1} & set(range(B))):
        if lens[b] == 0:
            assert not outs[0][b].any()
            continue
        ck, cv = build_oracle(k[b, :, :lens[b]], v[b, :, :lens[b]], stride_k=32, stride_v=8)
        assert_tight(outs[0][b], O.sdpa_fused(q[b], ck, cv, scale), what=f"b={b} len={lens[b]}")


@pytest.mark.parametrize("B,G,D,T", [(32, 4, 128, 1000), (256, 1, 64, 600)])
def test_without_a_workspace(B, G, D, T):
    # batches that fill the device with one workgroup per sequence need no
    # partials: without a workspace they are served whole, as the portable kernel's
    # (the same kernel at head_dim 64; at 128 its fp16 weights give the tight bar)
    from chronoquant_mlx_amd import ChronoQuantCache, _lib
    H, dev = 8, torch.device("cuda")
    g = torch.Generator(device="cuda")
    g.manual_seed(B)
    k, v = (torch.cumsum(torch.randn(B, H, T, D, device=dev, generator=g) * 0.1, 2).half() for _ in range(2))
    q = torch.randn(B, G * H, D, device=dev, generator=g).half()
    cache = ChronoQuantCache(stride_k=32, stride_v=8)
    cache.update_and_fetch(k, v)
    need = _lib.load().cq_decode_workspace_size(B, H, G * H, D, T)
    ws = torch.zeros(need, dtype=torch.uint8, device=dev)
    outs = []
    for fn, where, size in (("cq_decode_attn", None, 0), ("cq_decode_attn_generic", ws.data_ptr(), need)):
        out = torch.empty(B, G * H, D, device=dev)
        _lib.call(fn, cache._descriptor(), q.data_ptr(), _lib.CQ_F16, G * H, D ** -0.5, None, T, T,
                  out.data_ptr(), _lib.CQ_F32, where, size, _lib.stream_of(q))
        outs.append(out.cpu().numpy())
    if D == 64:
        assert np.array_equal(*outs)
    else:
        assert_tight(*outs, what="no workspace")
