"""The chunk append (append_bulk_kernel): its quotients against the oracle codec
on rows that put d / s at and around every point where a code changes, on
arbitrary bit patterns (zero rows, subnormals, infinities, NaN), and whole
appends against appends of 7 tokens at a time (the one-row kernels)."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _rows(dtype, kind, D=64):
    """int16 bit patterns [N, D]; in the "steps" rows the first value is the largest."""
    rng = np.random.default_rng(len(kind))
    if kind == "bits":
        return rng.integers(-32768, 32768, size=(4000, D)).astype(np.int16)
    mant = 10 if dtype == "f16" else 7
    one = 0x3c00 if dtype == "f16" else 0x3f80
    tops = [one + i for i in range(0, 1 << mant, 1 if dtype == "bf16" else 9)]
    tops += [1, 2, 3, 7, 50, 1000] if dtype == "f16" else [1, 0x2eff, 0x2f00, 0x2fdb, 0x7f7f]
    tops += [0x7bff] if dtype == "f16" else [0x7f00]
    out = []
    for top in tops:
        low = max(0, top - 6 * (1 << mant))  # down to top / 64
        d = np.arange(low, top + 1)
        d = rng.choice(d, size=min(len(d), 12 * (D - 1)), replace=False)
        d = np.concatenate([d, np.zeros((-len(d)) % (D - 1), np.int64)]) | (rng.integers(0, 2) << 15)
        d = d.reshape(-1, D - 1)
        out.append(np.concatenate([np.full((len(d), 1), top), d], axis=1))
    return np.concatenate(out).astype(np.uint16).view(np.int16)


@pytest.mark.parametrize("kind", ["steps", "bits"])
@pytest.mark.parametrize("dz", [0.0, 0.05, 1.0, 1.5])
@pytest.mark.parametrize("bits", [2, 3, 4])
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_codes_match_the_oracle(dtype, bits, dz, kind):
    from chronoquant_mlx_amd import ChronoQuantCache
    from chronoquant_mlx_amd.kernels import unpack_int4_codes
    rows = _rows(dtype, kind)
    N, D = rows.shape
    dt = torch.float16 if dtype == "f16" else torch.bfloat16
    x = torch.from_numpy(np.concatenate([np.zeros((1, D), np.int16), rows])).cuda().view(dt)[None, None]
    # a stride past the end: every row but the zero anchor is a residual
    cache = ChronoQuantCache(stride_k=1 << 23, stride_v=1 << 23, delta_bits_k=bits, delta_bits_v=bits,
                             dead_zone_k=dz, dead_zone_v=dz)
    cache.update_and_fetch(x, x)
    vals = x[0, 0, 1:].float().cpu().numpy()
    with np.errstate(all="ignore"):
        codes, scales = O.quantize_delta(vals.astype(np.float16) if dtype == "f16" else vals, bits, dz, dtype)
    got = unpack_int4_codes(cache.packed_codes_k[0, 0], D).cpu().numpy()
    assert np.array_equal(got, codes), np.argwhere(got != codes)[:5]
    gs = cache.pframe_scales_k[0, 0].cpu().numpy()
    nan = np.isnan(gs) & np.isnan(scales.reshape(-1))
    assert np.array_equal(gs.view(np.uint16)[~nan], scales.reshape(-1).view(np.uint16)[~nan])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,H,D,T,first,sk,sv,bk,bv,dense,token_major", [
    (2, 3, 64, 77, 0, 32, 8, 4, 4, False, False), (1, 2, 128, 130, 33, 5, 1, 3, 2, True, True),
    (2, 1, 256, 40, 20, 48, 24, 2, 3, True, False), (1, 2, 80, 65, 1, 64, 32, 4, 3, True, True),
    (1, 1, 8, 16, 0, 4, 4, 4, 4, False, False), (3, 2, 136, 100, 50, 12, 20, 4, 4, False, True),
    (1, 2, 72, 17, 0, 16, 16, 4, 4, False, False),
    # rows enough for the chunk kernel
    (4, 8, 64, 77, 0, 32, 8, 4, 4, False, False), (8, 16, 128, 130, 33, 5, 1, 3, 2, True, True),
    (2, 16, 256, 60, 20, 48, 24, 2, 3, True, False), (1, 40, 80, 65, 1, 64, 32, 4, 3, True, True),
    (4, 20, 8, 33, 0, 4, 4, 4, 4, False, False), (3, 20, 136, 100, 50, 12, 20, 4, 4, False, True),
    (4, 20, 72, 25, 0, 16, 16, 4, 4, False, False)])
def test_chunks_equal_short_appends(B, H, D, T, first, sk, sv, bk, bv, dense, token_major, dtype):
    from chronoquant_mlx_amd import ChronoQuantCache
    g = torch.Generator(device="cuda")
    g.manual_seed(D + T)
    k, v = (torch.cumsum(torch.randn(B, H, T, D, device="cuda", generator=g) * 0.2, 2).to(dtype) for _ in range(2))
    if token_major:
        k, v = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (k, v))
    states = []
    for sizes in ([first, T - first] if first else [T], [7] * (T // 7) + [T % 7]):
        cache = ChronoQuantCache(stride_k=sk, stride_v=sv, delta_bits_k=bk, delta_bits_v=bv, dead_zone_v=0.05,
                                 dense_residuals=dense)
        at = 0
        for n in sizes:
            cache.update_and_fetch(k[:, :, at:at + n], v[:, :, at:at + n])
            at += n
        states.append(cache.state)
    for i, (a, b) in enumerate(zip(*states)):
        view = torch.int16 if a.dtype == torch.float16 else torch.int32
        assert torch.equal(a.contiguous().view(view), b.contiguous().view(view)), i


@pytest.mark.parametrize("H", [2, 64])
def test_device_positions(H):
    # a chunk at per-sequence device offsets, one of them running past the
    # capacity: its rows past the end are dropped, the others unharmed
    from chronoquant_mlx_amd import ChronoQuantCache
    B, D, T, L = 3, 128, 256, 32
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    base, new = (torch.cumsum(torch.randn(B, H, n, D, device="cuda", generator=g) * 0.2, 2).half() for n in (T, L))
    start = [40, 3, T - 10]
    cache = ChronoQuantCache(stride_k=32, stride_v=8, capacity=T)
    cache.update_and_fetch(base, base)
    cap = cache._cap
    pos = torch.tensor(start, dtype=torch.int32, device="cuda")
    cache.bind_device_position(pos, cap)
    cache.update_and_fetch(new, new)
    cache.bind_device_position(None)
    assert cache._cap == cap
    for b, p in enumerate(start):
        ref = ChronoQuantCache(stride_k=32, stride_v=8, capacity=T)
        ref.update_and_fetch(base[b:b + 1], base[b:b + 1])
        ref.offset = p
        n = min(L, T - p)
        for s in range(n):
            ref.update_and_fetch(new[b:b + 1, :, s:s + 1], new[b:b + 1, :, s:s + 1])
        ref.offset = T
        for i, (x, y) in enumerate(zip(cache.state, ref.state)):
            view = torch.int16 if x.dtype == torch.float16 else torch.int32
            assert torch.equal(x[b].contiguous().view(view), y[0].contiguous().view(view)), (b, i)


@pytest.mark.parametrize("D,S,layout", [(128, 1, "plain"), (72, 1, "plain"), (128, 16, "plain"), (128, 1000, "plain"),
                                        (128, 1, "strided"), (128, 1, "beside"), (128, 1, "longer")])
def test_lengths_stored_by_the_append(D, S, layout):
    # one-row kernels, the four-row one and the chunk one; length vectors that the
    # append cannot store to (strided, longer than the batch) come from a separate sum
    from chronoquant_mlx_amd import ChronoQuantCache
    B = 3
    cache = ChronoQuantCache(stride_k=32, stride_v=8)
    cache.update_and_fetch(*(torch.randn(B, 2, 64, D, device="cuda").half() for _ in range(2)))
    n = B + 2 if layout == "longer" else B
    buf = torch.full((2 * n + 2,), -1, dtype=torch.int32, device="cuda")
    pos = buf[:n]
    lens = buf[n:2 * n] if layout != "strided" else torch.zeros(2 * n, dtype=torch.int32, device="cuda")[::2]
    if layout == "beside":
        pos, lens = torch.zeros(n, dtype=torch.int32, device="cuda"), torch.zeros(n, dtype=torch.int32, device="cuda")
    start = torch.tensor([5, 40, 17, 1, 2][:n], dtype=torch.int32, device="cuda")
    pos.copy_(start)
    cache.bind_device_position(pos, 128, lengths=lens)
    new = torch.randn(B, 2, S, D, device="cuda").half()
    cache.update_and_fetch(new, new)
    assert torch.equal(lens, start + S) and torch.equal(pos, start)
    if layout != "strided" and layout != "beside":
        assert buf[2 * n:].tolist() == [-1, -1]
