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

# fp32 output.  Both kernels sum products of fp32 weights in fp32 over up to 1300
# tokens: a few 2^-22 of the terms' size, which the outputs
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


def _rows64(comp, stride, T, D):
    """The cache's rows a + c * s of one oracle component [H, T, D], in 64 bits."""
    kf, pk, sc = comp.active()
    t = np.arange(T)
    x = kf.astype(np.float64)[:, t // stride]
    x[:, t % stride != 0] += O.unpack_int4(pk, D) * sc.astype(np.float64)[..., None]
    return x


@pytest.mark.parametrize("D,v_scale", [(64, 1.0), (256, 1.0), (256, 300.0), (96, 1e-4)])
@pytest.mark.parametrize("gap", [0.0, 5.0, 10.0, 15.0, 20.5, 30.0])
def test_weights_far_below_the_largest_keep_their_bits(gap, D, v_scale):
    # One token's score is about `gap` above all others and its V is 0, so the output is
    # made by the others' weights alone (v_scale 300: residual scales above 32).  Bar: p =
    # exp2(x - m) with x and m of up to 1.45 gap, each rounded twice to 2^-24 of itself,
    # and a few 2^-24 for exp2, the products and the sums (the v are of one sign, so
    # nothing cancels).
    from chronoquant_mlx_amd import ChronoQuantCache
    from chronoquant_mlx_amd.kernels import chronoquant_sdpa_cache_kernel as decode
    rng = np.random.default_rng(int(gap) + D)
    H, G, T, top = 2, 4, 600, 64  # (an anchor of both components: its V is 0 exactly)
    k = np.zeros((1, H, T, D), np.float16)
    k[..., 0] = 0.01 * rng.standard_normal((1, H, T))
    k[:, :, top, 0] = gap
    v = (v_scale * rng.uniform(0.5, 1.5, (1, H, T, D))).astype(np.float16)
    v[:, :, top] = 0
    cache = ChronoQuantCache(stride_k=32, stride_v=8, dead_zone_v=0.0)
    cache.update_and_fetch(to_gpu(k), to_gpu(v))
    q = np.zeros((1, G * H, D), np.float16)
    q[..., 0] = 1.0
    out = decode(to_gpu(q), cache, 1.0, out_dtype=torch.float32).cpu().numpy()[0]
    ck, cv = build_oracle(k[0], v[0], stride_k=32, stride_v=8)
    score = _rows64(ck, 32, T, D)[..., 0]
    w = np.exp(score - score.max(-1, keepdims=True))
    exact = np.einsum("ht,htd->hd", w, _rows64(cv, 8, T, D)) / w.sum(-1)[:, None]
    assert_close(out, np.repeat(exact, G, axis=0), 0.0, (gap + 2) * 2.0 ** -22, what=f"gap {gap}")


@pytest.mark.parametrize("D", [64, 256])
@pytest.mark.parametrize("t", [3, 8])
def test_infinite_values_like_the_portable_kernel(t, D):
    # a value past fp16's range makes its anchor (t = 8) or its row's scale infinite:
    # the dims it reaches are inf or NaN as there
    from chronoquant_mlx_amd import ChronoQuantCache
    from chronoquant_mlx_amd.kernels import chronoquant_sdpa_cache_kernel as decode
    rng = np.random.default_rng(t)
    k, v = (to_gpu(rng.standard_normal((1, 1, 9, D)), torch.bfloat16) for _ in range(2))
    v[0, 0, t, 5] = 3e38
    cache = ChronoQuantCache(stride_k=8, stride_v=8)
    cache.update_and_fetch(k, v)
    q = to_gpu(rng.standard_normal((1, 4, D)), torch.bfloat16)
    out, ref = (decode(q, cache, D ** -0.5, out_dtype=torch.float32, generic=g).cpu().numpy()
                for g in (False, True))
    assert np.isinf(ref[..., 5]).all()
    fin = np.isfinite(ref)
    assert np.array_equal(out[~fin], ref[~fin], equal_nan=True)
    if fin.any():  # (an infinite scale times a zero code: NaN in every other dim)
        assert_close(out[fin], ref[fin], ATOL, RTOL)


@pytest.mark.parametrize("D,G,top", [(64, 1, 33), (80, 4, 45), (256, 4, 60), (256, 8, 33)])
def test_bf16_queries_of_any_spread(D, G, top):
    # an element of 2^top meets keys that are 0 there: the scores come from the others,
    # far below fp16's range beside it
    from chronoquant_mlx_amd import ChronoQuantCache
    from chronoquant_mlx_amd.kernels import chronoquant_sdpa_cache_kernel as decode
    rng = np.random.default_rng(D + top)
    k, v = (rng.standard_normal((1, 2, 200, D)) for _ in range(2))
    k[..., D // 2] = 0
    cache = ChronoQuantCache(stride_k=32, stride_v=8)
    cache.update_and_fetch(to_gpu(k), to_gpu(v))
    q = rng.standard_normal((1, 2 * G, D))
    q[:, ::2, D // 2] = 2.0 ** top
    q = to_gpu(q, torch.bfloat16)
    out, ref = (decode(q, cache, 1.0, out_dtype=torch.float32, generic=g).cpu().numpy() for g in (False, True))
    assert_close(out, ref, ATOL, RTOL)
