"""The MFMA decode of head dims other than 128 and of dense rows
(cq_decode_wide.hip) against the oracle's fused semantics and the portable
kernel it takes over from: head dims around the K-step counts (32, 64, 96, 128,
256 and 8 more), splits with one token more than a unit, ragged batches with
empty sequences, q-head chunks, strides without a power of two, dense rows,
scales at fp16's ends, and the shapes that stay on the portable kernel."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.cqtest import assert_close, build_oracle, to_gpu

pytestmark = pytest.mark.gpu

# fp32 output.  Both kernels sum exact products (or products of 22-bit weights) in
# fp32 over up to 1300 tokens: a few 2^-22 of the terms' size, which the outputs
# (averages of values that drift to |v| ~ 4) do not cancel below a tenth of.
ATOL, RTOL = 2e-5, 1e-5


def _run(B, H, G, D, lens, dtype, sk, sv, bits=(4, 4), dense=False, v_scale=1.0):
    from chronoquant_mlx_amd import ChronoQuantCache
    from chronoquant_mlx_amd.kernels import chronoquant_sdpa_cache_kernel as decode
    rng = np.random.default_rng(D * 3 + G + sum(lens))
    T = max(lens)
    k, v = ((np.cumsum(rng.standard_normal((B, H, T, D)) * 0.1, axis=2) * s).astype(np.float16)
            for s in (1.0, v_scale))
    cache = ChronoQuantCache(stride_k=sk, stride_v=sv, delta_bits_k=bits[0], delta_bits_v=bits[1],
                             dead_zone_v=0.0, dense_residuals=dense)
    cache.update_and_fetch(to_gpu(k), to_gpu(v))
    q = to_gpu(rng.standard_normal((B, G * H, D)), torch.float16 if dtype == "f16" else torch.bfloat16)
    dl = torch.tensor(lens, dtype=torch.int32, device="cuda") if B > 1 else None
    scale = D ** -0.5
    out, again, ref = (decode(q, cache, scale, out_dtype=torch.float32, seq_lens=dl, generic=g).cpu().numpy()
                       for g in (False, False, True))
    assert np.array_equal(out, again)
    assert_close(out, ref, ATOL * v_scale, RTOL, what="portable kernel")
    if dtype == "f16" and not dense:
        for b in range(B):
            if lens[b] == 0:
                assert not out[b].any()
                continue
            ck, cv = build_oracle(k[b, :, :lens[b]], v[b, :, :lens[b]], stride_k=sk, stride_v=sv,
                                  bits_k=bits[0], bits_v=bits[1])
            fused = O.sdpa_fused(q[b].cpu().numpy(), ck, cv, scale)
            assert_close(out[b], fused, ATOL * v_scale, RTOL, what=f"oracle b={b}")


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("D", [32, 40, 64, 72, 96, 104, 120, 136, 192, 248, 256])
def test_head_dims(D, dtype):
    _run(1, 2, 4, D, [577], dtype, 32, 8)


@pytest.mark.parametrize("B,H,G,D,lens,sk,sv", [
    (1, 2, 4, 256, [1], 32, 8), (1, 1, 1, 256, [512], 32, 8), (1, 3, 8, 64, [513], 4, 4),
    (5, 2, 4, 256, [1300, 0, 1, 512, 65], 32, 8), (3, 1, 20, 96, [700, 64, 63], 12, 20),
    (2, 8, 4, 80, [1025, 300], 48, 24)])
def test_lengths_heads_and_strides(B, H, G, D, lens, sk, sv):
    _run(B, H, G, D, lens, "f16", sk, sv)


@pytest.mark.parametrize("D,G,sk,sv,bits", [(256, 4, 64, 32, (4, 3)), (128, 8, 48, 24, (3, 2)),
                                            (80, 4, 16, 16, (2, 3)), (64, 1, 4, 8, (3, 4))])
def test_dense_rows(D, G, sk, sv, bits):
    _run(2, 2, G, D, [700, 333], "bf16", sk, sv, bits, dense=True)


@pytest.mark.parametrize("v_scale", [3000.0, 1e-3])
def test_value_scales(v_scale):
    # residual scales up to ~100 (above the weights' headroom, which the chunk's
    # largest scale then lowers) and fp16-subnormal ones
    _run(1, 2, 4, 256, [600], "f16", 32, 8, v_scale=v_scale)


@pytest.mark.parametrize("D,dtype,sk", [(24, "f16", 8), (36, "f16", 8), (64, "f32", 8), (64, "f16", 3)])
def test_shapes_left_to_the_portable_kernel(D, dtype, sk):
    from chronoquant_mlx_amd import ChronoQuantCache
    from chronoquant_mlx_amd.kernels import chronoquant_sdpa_cache_kernel as decode
    rng = np.random.default_rng(D)
    cache = ChronoQuantCache(stride_k=sk, stride_v=8)
    cache.update_and_fetch(*(to_gpu(rng.standard_normal((1, 2, 90, D))) for _ in range(2)))
    q = to_gpu(rng.standard_normal((1, 4, D)), torch.float32 if dtype == "f32" else torch.float16)
    out, ref = (decode(q, cache, D ** -0.5, generic=g) for g in (False, True))
    assert torch.equal(out, ref)
