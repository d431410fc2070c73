"""cq_flash_attn against the oracle's restatement of the reconstruct fallback
(attention.py:8-20, 61-74): head dims on both sides of the padded sizes, row
tiles and key blocks with remainders, split keys, boolean masks of every
broadcast form (rows that see no key among them), dense rows, fp16 and bf16
queries, and the calls it leaves to the fallback."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.cqtest import assert_close, build_gpu_cache, build_oracle, to_gpu

pytestmark = pytest.mark.gpu


def _stream(rng, B, H, T, D):
    return np.cumsum(rng.standard_normal((B, H, T, D)) * 0.1, axis=2).astype(np.float16)


def _mask(kind, rng, L, T):
    """(mask as [L, T] booleans or None, what the call takes)."""
    if kind in ("causal", None):
        return None, kind
    if kind == "window":
        q, k = np.arange(T - L, T)[:, None], np.arange(T)[None]
        m = (q >= k) & (q < k + max(1, T // 4))
    elif kind == "rows":  # one column for every key: broadcast over the keys
        return np.broadcast_to(rng.random((L, 1)) > 0.5, (L, T)), None
    else:
        m = rng.random((L, T)) > 0.5
        m[0] = False  # a row that sees nothing weighs every key alike
    return m, torch.from_numpy(m).cuda()


# (H, G, D, T, L, mask, params): 64-, 96-, 128- and 256-wide rows and their edges
# (8, 72, 80, 136), key blocks of 32 and 64 with one key more or less, 256-row
# tiles with one row more (G L = 256, 257), and enough keys to split
CASES = [
    (2, 4, 64, 65, 64, "causal", {}), (2, 3, 72, 300, 77, "causal", {}), (1, 2, 80, 127, 128 - 1, None, {}),
    (2, 1, 8, 40, 3, "causal", {}), (1, 4, 136, 33, 33, "causal", {}), (2, 4, 256, 1000, 64, "causal", {}),
    (1, 1, 256, 32, 1, None, {}), (1, 1, 256, 2049, 257, "random", {}), (2, 4, 128, 1000, 65, "window", {}),
    (1, 4, 128, 129, 129, "random", {}), (1, 2, 96, 64, 20, "rows", {}), (1, 4, 256, 500, 100, "window", {}),
    (2, 4, 128, 600, 50, "causal", dict(stride_k=64, stride_v=32, bits_v=3, dz_v=0.05, dense=True)),
    (1, 2, 80, 200, 30, "causal", dict(stride_k=5, stride_v=1, bits_k=2, dense=True)),
]


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("H,G,D,T,L,mask,params", CASES)
def test_flash_matches_fallback(H, G, D, T, L, mask, params, dtype):
    from chronoquant_mlx_amd import ChronoQuantCache, kernels
    rng = np.random.default_rng(D * 7 + T + L)
    k, v = _stream(rng, 1, H, T, D), _stream(rng, 1, H, T, D)
    p = dict(dict(stride_k=32, stride_v=8), **params)
    dense = p.pop("dense", False)
    cache = ChronoQuantCache(stride_k=p["stride_k"], stride_v=p["stride_v"], delta_bits_k=p.get("bits_k", 4),
                             delta_bits_v=p.get("bits_v", 4), dead_zone_v=p.get("dz_v", 0.0),
                             dense_residuals=dense)
    cache.update_and_fetch(to_gpu(k), to_gpu(v))
    q32 = rng.standard_normal((1, G * H, L, D)).astype(np.float32)
    scale = D ** -0.5
    m, arg = _mask(mask, rng, L, T)
    if m is not None and arg is None:
        arg = torch.from_numpy(m[:, :1].copy()).cuda()
    ck, cv = build_oracle(k[0], v[0], **p)
    rk, rv = ck.reconstruct(), cv.reconstruct()
    dt = torch.float16 if dtype == "f16" else torch.bfloat16
    qt = to_gpu(q32, dt)
    out = kernels.chronoquant_flash_kernel(qt, cache, scale, arg)
    assert out is not None and out.dtype == dt
    if dtype == "f16":
        ref = O.sdpa_fallback(qt.cpu().numpy()[0], rk, rv, scale, causal=mask == "causal", mask=m)
    else:
        bits = qt.cpu().view(torch.int16).numpy().view(np.uint16)[0]
        ref = O.bf16_to_f32(O.sdpa_fallback_bf16q(bits, rk, rv, scale, causal=mask == "causal", mask=m))
    assert_close(out.float().cpu().numpy()[0], ref.astype(np.float64), what=f"{dtype} {mask}")


def _cancelling_scores(depth):
    """(a, b): two fp16 scores about `depth` below 0 whose weights differ by 2^-5 and,
    held in fp16 alone (the largest weight at 2^14), are off by most of half a place
    each in opposite directions."""
    c = -depth - np.arange(0, 2000) * 2.0 ** -10
    c = np.unique(c.astype(np.float16).astype(np.float64))
    p = np.exp(c)
    if depth > 20:  # (below fp16's range beside the largest: any will do)
        return c[-1], c[np.argmin(np.abs(c[-1] - c - 2.0 ** -5))]
    off = (p * 2.0 ** 14).astype(np.float16).astype(np.float64) * 2.0 ** -14 / p - 1
    for x in np.argsort(-off):
        near = np.flatnonzero(np.abs(c[x] - c - 2.0 ** -5) < 2.0 ** -6)
        if near.size and off[near].min() < -0.7 * off[x]:
            return c[x], c[near[np.argmin(off[near])]]


@pytest.mark.parametrize("depth", [2, 8, 14, 20, 40, 60])
@pytest.mark.parametrize("D", [64, 80, 128, 256])
def test_flash_bf16_weights_keep_32_bits(D, depth):
    # A dominant key of V = 0, then 200 keys of V = 1 and 200 of V = -1 whose weights
    # nearly cancel: the output is 2^-5 of what either group makes.  Bar: the output's
    # rounding to bf16 (2^-8), and 2^5 times the weights' error in fp32 arithmetic (scores
    # of up to 87 in binary orders, each rounded to 2^-24 of itself: 2^-17).  Weights held
    # in fp16 miss it, and so do fp16 pairs (23 bits, down to 2^-24 beside a largest
    # weight of 2^14) from a depth of 20 on.
    from chronoquant_mlx_amd import ChronoQuantCache, kernels
    n = 200
    a, b = _cancelling_scores(depth)
    score = np.concatenate([[0.0], np.full(n, a), np.full(n, b)])
    value = np.concatenate([[0.0], np.ones(n), -np.ones(n)])
    order = np.concatenate([[0], 1 + np.random.default_rng(depth).permutation(2 * n)])
    score, value = score[order], value[order]
    w = np.exp(score)
    exact = (w * value).sum() / w.sum()
    bar = (2.0 ** -8 + 2.0 ** -12) * abs(exact)
    hi = (w * 2.0 ** 14).astype(np.float16).astype(np.float64)
    lo = (w * 2.0 ** 14 - hi).astype(np.float16).astype(np.float64)
    for kept, enough in ((hi, False), (hi + lo, depth < 20)):
        assert (abs((kept * value).sum() / (w.sum() * 2.0 ** 14) - exact) < bar) == enough
    k, v = np.zeros((1, 1, 2 * n + 1, D), np.float16), np.zeros((1, 1, 2 * n + 1, D), np.float16)
    k[0, 0, :, 0], v[0, 0] = score, value[:, None]
    cache = ChronoQuantCache(stride_k=1, stride_v=1)
    cache.update_and_fetch(to_gpu(k), to_gpu(v))
    q = torch.zeros(1, 2, 2, D, dtype=torch.bfloat16, device="cuda")
    q[..., 0] = 1.0
    out = kernels.chronoquant_flash_kernel(q, cache, 1.0, None).double().cpu().numpy()
    assert np.all(np.abs(out - exact) <= bar), (out.ravel()[0], exact)


@pytest.mark.parametrize("shape", [(1, 1, 1, 9, 70), (1, 2, 1, 9, 70), (2, 2, 3, 9, 70), (9, 1), (70,)])
def test_flash_mask_broadcasts_like_the_fallback(shape):
    from chronoquant_mlx_amd import attention as A
    B, H, G, L, T, D = 2, 2, 3, 9, 70, 128
    rng = np.random.default_rng(len(shape))
    cache = build_gpu_cache(_stream(rng, B, H, T, D), _stream(rng, B, H, T, D), stride_k=32, stride_v=8)
    q = to_gpu(rng.standard_normal((B, G * H, L, D)))
    mask = torch.from_numpy(rng.random(shape) > 0.4).cuda()
    got = A.chronoquant_sdpa(q, None, None, cache, D ** -0.5, mask)
    A.PREFILL_KERNEL = False
    try:
        ref = A.chronoquant_sdpa(q, None, None, cache, D ** -0.5, mask)
    finally:
        A.PREFILL_KERNEL = True
    assert_close(got.float().cpu().numpy(), ref.float().cpu().numpy())


@pytest.mark.parametrize("G,D,L,T", [(4, 128, 77, 2100), (7, 64, 40, 333), (1, 256, 300, 1025), (16, 96, 65, 1500)])
@pytest.mark.parametrize("kind", ["window", "padded", "one key", "blind row", "per head", "per sequence"])
def test_flash_passes_over_hidden_blocks(kind, G, D, L, T):
    # masks that hide whole key blocks from whole row tiles, alike for every
    # head or not; one row that sees nothing brings every block of its tile back
    from chronoquant_mlx_amd import attention as A
    B, H = 2, 2
    rng = np.random.default_rng(G)
    cache = build_gpu_cache(_stream(rng, B, H, T, D), _stream(rng, B, H, T, D), stride_k=32, stride_v=8)
    q = to_gpu(rng.standard_normal((B, G * H, L, D)))
    i, t = torch.arange(T - L, T, device="cuda")[:, None], torch.arange(T, device="cuda")[None]
    window = (i >= t) & (i < t + T // 5)
    mask = {"window": window, "padded": (t >= T // 3) & (i >= t), "one key": t == (i * 7) % T,
            "blind row": window & (i != T - 2),
            "per head": window & (t % G == torch.arange(G, device="cuda").view(1, 1, G, 1, 1)),
            "per sequence": (i >= t) & (t >= 300 * torch.arange(B, device="cuda").view(B, 1, 1, 1, 1))}[kind]
    got = A.chronoquant_sdpa(q, None, None, cache, D ** -0.5, mask)
    A.PREFILL_KERNEL = False
    try:
        ref = A.chronoquant_sdpa(q, None, None, cache, D ** -0.5, mask)
    finally:
        A.PREFILL_KERNEL = True
    assert_close(got.float().cpu().numpy(), ref.float().cpu().numpy())


def test_flash_leaves_to_the_fallback():
    # additive masks, fp32 queries, head dims that are no multiple of 8, causal
    # chunks longer than the cache, and queries that autograd follows
    from chronoquant_mlx_amd import chronoquant_sdpa, kernels
    rng = np.random.default_rng(1)
    H, L, T = 2, 5, 40
    for D, dt, mask in ((64, torch.float16, torch.zeros(L, T, device="cuda")), (64, torch.float32, None),
                        (12, torch.float16, None), (64, torch.float16, "grad")):
        cache = build_gpu_cache(_stream(rng, 1, H, T, D), _stream(rng, 1, H, T, D), stride_k=32, stride_v=8)
        q = to_gpu(rng.standard_normal((1, H, L, D)), dt)
        if isinstance(mask, str):
            q.requires_grad_(True)
            mask = torch.ones(L, T, dtype=torch.bool, device="cuda")
        assert kernels.chronoquant_flash_kernel(q, cache, 1.0, mask) is None
        out = chronoquant_sdpa(q, None, None, cache, D ** -0.5, mask)
        assert out.shape == q.shape and bool(torch.isfinite(out).all())
        assert out.requires_grad == q.requires_grad
    q = to_gpu(rng.standard_normal((1, H, T + 1, 12)))
    assert kernels.chronoquant_flash_kernel(q, cache, 1.0, "causal") is None


@pytest.mark.parametrize("D,top", [(64, 33), (80, 45), (128, 60), (256, 33)])
def test_flash_bf16_queries_of_any_spread(D, top):
    # an element of 2^top meets keys that are 0 there: the scores come from the others,
    # far below fp16's range beside it.  Against the fallback (fp32 products), one
    # rounding of the output to bf16 apart.
    from chronoquant_mlx_amd import chronoquant_sdpa, kernels
    from chronoquant_mlx_amd import attention as A
    rng = np.random.default_rng(D + top)
    k, v = (rng.standard_normal((1, 2, 200, D)) for _ in range(2))
    k[..., D // 2] = 0
    cache = build_gpu_cache(k, v, stride_k=32, stride_v=8)
    q = rng.standard_normal((1, 8, 9, D))
    q[:, ::2, :, D // 2] = 2.0 ** top
    q = to_gpu(q, torch.bfloat16)
    got = kernels.chronoquant_flash_kernel(q, cache, D ** -0.5, "causal")
    A.PREFILL_KERNEL = False
    try:
        ref = chronoquant_sdpa(q, None, None, cache, D ** -0.5, "causal")
    finally:
        A.PREFILL_KERNEL = True
    assert_close(got.float().cpu().numpy(), ref.float().cpu().numpy(), 1e-3, 2.0 ** -7)


def test_flash_masks_under_vmap():
    # a mask that a transform follows has no storage of its own: torch ops, as before
    from chronoquant_mlx_amd import chronoquant_sdpa
    rng = np.random.default_rng(0)
    cache = build_gpu_cache(_stream(rng, 1, 2, 40, 64), _stream(rng, 1, 2, 40, 64), stride_k=32, stride_v=8)
    q = to_gpu(rng.standard_normal((1, 4, 5, 64)))
    masks = torch.from_numpy(rng.random((3, 5, 40)) > 0.4).cuda()
    out = torch.vmap(lambda m: chronoquant_sdpa(q, None, None, cache, 0.125, m))(masks)
    for i in range(3):
        ref = chronoquant_sdpa(q, None, None, cache, 0.125, masks[i])
        assert_close(out[i].float().cpu().numpy(), ref.float().cpu().numpy())


def _both(q, cache, scale, mask):
    from chronoquant_mlx_amd import chronoquant_sdpa, kernels
    from chronoquant_mlx_amd import attention as A
    got = kernels.chronoquant_flash_kernel(q, cache, scale, mask)
    A.PREFILL_KERNEL = False
    try:
        ref = chronoquant_sdpa(q, None, None, cache, scale, mask)
    finally:
        A.PREFILL_KERNEL = True
    return got.float().cpu().numpy(), ref.float().cpu().numpy()


@pytest.mark.parametrize("D,T", [(64, 300), (128, 700), (256, 300)])
@pytest.mark.parametrize("peak", [224.0, 255.8, 300.0])
@pytest.mark.parametrize("kind", ["causal", "window", "half"])
def test_flash_scores_at_the_lowest_value(kind, peak, D, T):
    # fp16 scores of the visible keys about peak^2 below 0: clear of fp16's lowest
    # value, which hidden keys' scores have, next to it, and past it (-inf), where the
    # hidden keys take the weight.  Rows that see every key at -inf are NaN.  (window
    # and half hide whole key blocks.)
    L = 40
    rng = np.random.default_rng(D)
    k = np.zeros((1, 2, T, D))
    k[..., 0] = peak + 0.125 * rng.integers(-1, 2, size=(1, 2, T))
    cache = build_gpu_cache(k, _stream(rng, 1, 2, T, D), stride_k=1, stride_v=8)
    q = torch.zeros(1, 4, L, D, dtype=torch.float16, device="cuda")
    q[..., 0] = -peak
    i, t = torch.arange(T - L, T, device="cuda")[:, None], torch.arange(T, device="cuda")[None]
    mask = {"causal": "causal", "window": (i >= t) & (i < t + 90), "half": (t >= T // 2) & (i >= -t)}[kind]
    if D == 128 and kind == "causal":
        mask = i >= t  # (the string takes the head_dim-128 kernel in chronoquant_sdpa)
    got, ref = _both(q, cache, 1.0, mask)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert_close(np.nan_to_num(got), np.nan_to_num(ref))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [64, 80, 256])
@pytest.mark.parametrize("mask", [None, "causal", "window"])
def test_flash_infinite_values_like_the_fallback(mask, D, dtype):
    # V past fp16's range at an anchor (infinite) of some keys: +-inf where a row gives
    # it weight, NaN where the weight is 0 (a hidden key) or the signs differ, and the
    # other dims as ever.  Few keys, so that no weight rounds to 0.
    T, L = 150, 70
    rng = np.random.default_rng(D)
    k, v = (to_gpu(0.3 * rng.standard_normal((1, 2, T, D)), torch.bfloat16) for _ in range(2))
    v[0, 0, 148, 3], v[0, 0, 64, 5], v[0, 1, 4, 6], v[0, 1, 140, 6] = 3e38, -3e38, 3e38, -3e38
    cache = build_gpu_cache(k.float().cpu().numpy(), v.float().cpu().numpy(), stride_k=4, stride_v=1,
                            dtype=torch.bfloat16)
    q = to_gpu(0.3 * rng.standard_normal((1, 8, L, D)), dtype)
    i, t = torch.arange(T - L, T, device="cuda")[:, None], torch.arange(T, device="cuda")[None]
    got, ref = _both(q, cache, D ** -0.5, (i >= t) & (i < t + 30) if mask == "window" else mask)
    assert np.isnan(ref).any() and (mask == "window" or np.isinf(ref).any())
    fin = np.isfinite(ref)
    assert np.array_equal(got[~fin], ref[~fin], equal_nan=True)
    assert_close(got[fin], ref[fin])


@pytest.mark.parametrize("dtype,mask", [(torch.float16, "causal"), (torch.bfloat16, "window")])
def test_flash_splits_over_several_rounds(dtype, mask):
    # more tiles than CUs and splits all the same, so that the workgroups run in
    # several rounds; against the fallback, a kv head at a time
    from chronoquant_mlx_amd import _lib, kernels
    B, H, G, D, T, L = 1, 8, 4, 64, 8192, 2560
    g = torch.Generator(device="cuda")
    g.manual_seed(1)
    k, v = (torch.cumsum(0.1 * torch.randn(B, H, T, D, device="cuda", generator=g), 2).half() for _ in range(2))
    q = torch.randn(B, G * H, L, D, device="cuda", generator=g).to(dtype)
    cache = build_gpu_cache(k.cpu().numpy(), v.cpu().numpy(), stride_k=32, stride_v=8)
    need = _lib.load().cq_flash_scratch_size(cache._descriptor(), G * H, L, T)
    assert G * L // 256 * H * B > torch.cuda.get_device_properties(0).multi_processor_count
    assert need > 2 * B * H * T * D * 2 + 2 * (B * G * H * L) * D * 4  # two splits' partials
    i, t = torch.arange(T - L, T, device="cuda")[:, None], torch.arange(T, device="cuda")[None]
    m = (i >= t) & (i < t + 3000) if mask == "window" else mask
    got = kernels.chronoquant_flash_kernel(q, cache, D ** -0.5, m)
    for h in range(0, H, 7):
        part = build_gpu_cache(k[:, h:h + 1].cpu().numpy(), v[:, h:h + 1].cpu().numpy(), stride_k=32, stride_v=8)
        _, ref = _both(q[:, G * h:G * h + G].contiguous(), part, D ** -0.5, m)
        assert_close(got[:, G * h:G * h + G].float().cpu().numpy(), ref)
