"""Operand ranges of the MFMA attention kernels. Their operands are fp16 (normal from 2^-14 to
65504) while the reference computes in fp32 (``laguna_mlx/q8_attn.py:117``): the kernels scale q
and the P.V operand (softmax weight times V scale) by powers of two chosen from the data, so
queries far outside fp16's range and V groups with tiny or huge scales keep fp32-level accuracy.

Each case against the fused-arithmetic oracle (fp32 dequantize, float64 softmax) at the parity
bar scaled to the inputs: max-abs 2e-3 x (V std) + rel 1e-2. Peaked scores (large q) make the
output rest on a handful of keys, where a coarse P.V operand shows most.
"""
import numpy as np
import pytest
import torch

from gpu_util import RTOL, assert_attn_close, cache_np, make_cache, to_dev_bf16
from oracle import attention as A
from oracle import quantize as Q

pytestmark = pytest.mark.gpu

# (q std, V std): huge and tiny queries, V groups with tiny and huge scales, peaked softmax
RANGES = [(1e4, 1.0), (2e5, 1.0), (1e-4, 1.0), (1.0, 0.01), (3.0, 0.005), (3.0, 1e-4),
          (1.0, 1e3), (3.0, 1e5), (30.0, 0.02)]


def _case(dev, seed, B, Hkv, n, bits, qstd, vstd, G, L):
    rng = np.random.default_rng(seed)
    cap = (n + 255) // 256 * 256 + 256
    kq, vq = make_cache(rng, B, Hkv, n, cap, dev, bits=bits, vstd=vstd)
    q = Q.round_bf16(Q.randn_bf16(rng, (B, Hkv * G, L, 128)) * np.float32(qstd))
    return kq, vq, q


# (bits, G, B) -> the kernel that runs: one 8-bit sequence of at most 65,536 rows takes the
# dense kernel (attn_dense.hip) whatever G; a batch of 8-bit sequences with G <= 4 takes the
# packed kernel (qattn.hip); the 4-bit cache always takes its packed kernel (attn_q4.hip)
DECODE_KERNELS = {(8, 4, 1): "dense", (8, 1, 1): "dense", (8, 6, 1): "dense",
                  (8, 4, 2): "8-bit packed", (8, 1, 2): "8-bit packed", (4, 4, 1): "4-bit packed"}


@pytest.mark.parametrize("qstd,vstd", RANGES)
@pytest.mark.parametrize("bits,G,B", list(DECODE_KERNELS))
def test_decode_operand_range(dev, qstd, vstd, bits, G, B):
    """Decode on each kernel (DECODE_KERNELS); a batch of two sequences of 9,000 and 7,777 rows
    for the packed 8-bit kernel, each sequence checked."""
    from lagunalab_amd.q8_attn import decode_attention
    n = 9000
    lens = [n, 7777][:B]
    kq, vq, q = _case(dev, int(qstd * 7 + vstd * 13) % 1000 + G + bits + 100 * B, B, 8, n, bits,
                      qstd, vstd, G, 1)
    got = decode_attention(to_dev_bf16(q, dev), kq, vq, lens=lens, scale=128 ** -0.5)
    assert torch.isfinite(got.float()).all()
    for b in range(B):
        sl = slice(b, b + 1)
        want = A.fused_attention(q[sl], cache_np(tuple(t[sl] for t in kq)),
                                 cache_np(tuple(t[sl] for t in vq)), lens[b], 128 ** -0.5,
                                 bits=bits)
        assert_attn_close(got[sl], want, f"{DECODE_KERNELS[bits, G, B]} {bits}-bit G={G} "
                          f"sequence {b} q std {qstd} V std {vstd}", 2e-3 * vstd, RTOL)


@pytest.mark.parametrize("qstd,vstd", RANGES)
def test_verify_operand_range(dev, qstd, vstd):
    """The 5-row causal verify block (dense kernel, 20 rows per KV head)."""
    from lagunalab_amd.q8_attn import q8_verify_attention
    n = 6001
    kq, vq, q = _case(dev, int(qstd * 3 + vstd * 5) % 1000, 1, 8, n, 8, qstd, vstd, 4, 5)
    got = q8_verify_attention(to_dev_bf16(q, dev), kq, vq, n, 128 ** -0.5)
    assert torch.isfinite(got.float()).all()
    want = A.fused_attention(q, cache_np(kq), cache_np(vq), n, 128 ** -0.5, causal=True)
    assert_attn_close(got, want, f"verify q std {qstd} V std {vstd}", 2e-3 * vstd, RTOL)


@pytest.mark.parametrize("B", [1, 2], ids=["dense", "packed"])
def test_v_scales_changing_across_the_cache(dev, B):
    """V groups whose scales jump by 2^10 and 2^20 between 700-row regions of the cache: the P.V
    factor is re-chosen up and down as a wave's super-tiles cross the regions (rescaling what it
    accumulated). The keys of the smallest-scale region get the largest scores, so the output
    rests on the values that are 2^20 below the others. One sequence runs the dense kernel; a
    batch of two (the same cache contents, 12,000 and 10,650 rows) the packed 8-bit kernel."""
    from lagunalab_amd.q8_attn import decode_attention
    from lagunalab_amd.quant import quantize_into
    rng = np.random.default_rng(77)
    n, cap, Hkv, G = 12000, 12288, 8, 4
    lens = [n, 10650][:B]
    region = (np.arange(n) // 700) % 3  # V std 1, 2^-20, 2^-10
    # the G query heads of a KV head: one direction plus a little noise
    q = Q.randn_bf16(rng, (1, Hkv, 1, 1, 128)) * np.float32(4.0)
    q = Q.round_bf16(q + 0.3 * Q.randn_bf16(rng, (1, Hkv, G, 1, 128))).reshape(1, Hkv * G, 1, 128)
    qdir = q[0, ::G, 0] / np.linalg.norm(q[0, ::G, 0], axis=-1, keepdims=True)  # [Hkv, 128]
    shift = np.where(region == 1, 6.0, -6.0).astype(np.float32)
    k = Q.randn_bf16(rng, (1, Hkv, n, 128)) + shift[None, None, :, None] * qdir[None, :, None, :]
    v = Q.randn_bf16(rng, (1, Hkv, n, 128)) * (np.float32(2.0) ** np.array([0, -20, -10])[region]
                                                 ).astype(np.float32)[None, None, :, None]
    caches = []
    for x in (k, v):
        c = (torch.zeros((B, Hkv, cap, 128), dtype=torch.uint8, device=dev),
             torch.zeros((B, Hkv, cap, 2), dtype=torch.bfloat16, device=dev),
             torch.zeros((B, Hkv, cap, 2), dtype=torch.bfloat16, device=dev))
        xb = np.repeat(Q.round_bf16(x), B, axis=0)
        quantize_into(to_dev_bf16(xb, dev), *c, 0, 64, 8)
        caches.append(c)
    qb = np.repeat(q, B, axis=0)
    got = decode_attention(to_dev_bf16(qb, dev), caches[0], caches[1], lens=lens,
                           scale=128 ** -0.5)
    for b in range(B):
        sl = slice(b, b + 1)
        want = A.fused_attention(q, cache_np(tuple(t[sl] for t in caches[0])),
                                 cache_np(tuple(t[sl] for t in caches[1])), lens[b], 128 ** -0.5)
        mag = float(np.abs(want).max())
        assert mag < 2.0 ** -14, mag  # the output is the small-scale region's
        assert_attn_close(got[sl], want, f"V scales jumping by 2^10 and 2^20, sequence {b}",
                          2e-3 * mag, RTOL)


# ------------------------------------------------------------------------------------- prefill
# For groupings other than 1, 2, 4 and 8 the prefill kernel keeps the verify kernel's arithmetic: exact
# codes as operands, the affine terms in 32 bits, P times the V scale in fp16 (2^-11 relative) with a
# power-of-two factor per quant group and 64-key tile. The bars of the next two tests, from the operands'
# 2^-11 steps (a score of size s moving by s 2^-11), leave it room.

@pytest.mark.parametrize("G", [6, 3])
@pytest.mark.parametrize("qstd,kstd,vstd", [(1e-4, 1.0, 1.0), (1.0, 1.0, 1e-6), (1.0, 1.0, 1e5),
                                            (2e5, 1e-5, 1.0), (1e-4, 3e5, 1.0), (2e5, 1e-5, 1e6),
                                            (3.0, 1e-3, 1e-4)])
def test_prefill_operand_range(dev, G, qstd, kstd, vstd):
    """A 37-row chunk behind 963 rows: q, K and V far outside fp16's range on either side."""
    from lagunalab_amd.q8_attn import q8_prefill_attention
    rng = np.random.default_rng(int(qstd * 3 + vstd * 5) % 1000 + G)
    n, L, Hkv, cap = 1000, 37, 2, 1024
    caches = []
    for std in (kstd, vstd):
        x = Q.round_bf16(Q.randn_bf16(rng, (1, Hkv, n, 128)) * np.float32(std))
        from lagunalab_amd.quant import quantize_into
        c = (torch.zeros((1, Hkv, cap, 128), dtype=torch.uint8, device=dev),
             torch.zeros((1, Hkv, cap, 2), dtype=torch.bfloat16, device=dev),
             torch.zeros((1, Hkv, cap, 2), dtype=torch.bfloat16, device=dev))
        quantize_into(to_dev_bf16(x, dev), *c, 0, 64, 8)
        caches.append(c)
    q = Q.round_bf16(Q.randn_bf16(rng, (1, Hkv * G, L, 128)) * np.float32(qstd))
    got = q8_prefill_attention(to_dev_bf16(q, dev), *caches, n, 128 ** -0.5)
    assert torch.isfinite(got.float()).all()
    want = A.fused_attention(q, cache_np(caches[0]), cache_np(caches[1]), n, 128 ** -0.5,
                             causal=True)
    s = max(1.0, qstd * kstd)  # largest scores ~5 s nats, each off by up to 2^-11 of its terms
    assert_attn_close(got, want, f"prefill G={G} q {qstd} K {kstd} V {vstd}", 2e-3 * s * vstd, RTOL)


@pytest.mark.parametrize("G", [6, 3])
def test_prefill_factors_change_between_tiles(dev, G):
    """K and V whose sizes jump by powers of two between 300-row regions (so that tiles straddle
    them): the V factor rises and falls. The keys of the smallest-V region get the largest scores.
    (V sizes 2^-20 apart: where a tile straddles the regions, P times the small V scales is 2^-16 or
    less of fp16's range, steps of 2^-9 of its largest value.)"""
    from lagunalab_amd.q8_attn import q8_prefill_attention
    from lagunalab_amd.quant import quantize_into
    rng = np.random.default_rng(78)
    n, cap, Hkv, L = 3000, 3072, 2, 70
    region = (np.arange(n) // 300) % 3
    q = Q.randn_bf16(rng, (1, Hkv, 1, 1, 128)) * np.float32(4.0)
    q = Q.round_bf16(q + 0.3 * Q.randn_bf16(rng, (1, Hkv, G, L, 128))).reshape(1, Hkv * G, L, 128)
    qdir = q[0, ::G, 0] / np.linalg.norm(q[0, ::G, 0], axis=-1, keepdims=True)
    shift = np.where(region == 1, 6.0, -6.0).astype(np.float32)
    k = Q.randn_bf16(rng, (1, Hkv, n, 128)) + shift[None, None, :, None] * qdir[None, :, None, :]
    k[:, :, region == 2] *= np.float32(2.0 ** -12)
    v = Q.randn_bf16(rng, (1, Hkv, n, 128)) * (np.float32(2.0) ** np.array([5, -15, -5])[region]
                                               ).astype(np.float32)[None, None, :, None]
    caches = []
    for x in (k, v):
        c = (torch.zeros((1, Hkv, cap, 128), dtype=torch.uint8, device=dev),
             torch.zeros((1, Hkv, cap, 2), dtype=torch.bfloat16, device=dev),
             torch.zeros((1, Hkv, cap, 2), dtype=torch.bfloat16, device=dev))
        quantize_into(to_dev_bf16(Q.round_bf16(x), dev), *c, 0, 64, 8)
        caches.append(c)
    got = q8_prefill_attention(to_dev_bf16(q, dev), *caches, n, 128 ** -0.5)
    want = A.fused_attention(q, cache_np(caches[0]), cache_np(caches[1]), n, 128 ** -0.5,
                             causal=True)
    assert torch.isfinite(got.float()).all()
    # each row against its own largest value: the rows rest on different regions
    mag = np.abs(want).max(-1, keepdims=True)
    err = np.abs(got.float().cpu().numpy() - want)
    assert np.all(err <= 8e-3 * mag + RTOL * np.abs(want)), float((err / mag).max())


def _buffers(dev, x, cap):
    """x [1, H, n, 128] quantized into full-capacity 8-bit buffers."""
    from lagunalab_amd.quant import quantize_into
    H = x.shape[1]
    c = (torch.zeros((1, H, cap, 128), dtype=torch.uint8, device=dev),
         torch.zeros((1, H, cap, 2), dtype=torch.bfloat16, device=dev),
         torch.zeros((1, H, cap, 2), dtype=torch.bfloat16, device=dev))
    quantize_into(to_dev_bf16(Q.round_bf16(x), dev), *c, 0, 64, 8)
    return c


def _split(n, L, G, Hkv):
    from lagunalab_amd import _lib
    return _lib.load().lq_prefill_workspace_bytes(1, Hkv * G, Hkv, L, n) > 0


@pytest.mark.parametrize("G,n,L,Hkv", [(6, 1000, 100, 2), (6, 8193, 256, 2), (3, 3000, 200, 2),
                                       (12, 3000, 100, 1)])
def test_prefill_of_other_groupings_is_as_exact_as_the_verify_kernel(dev, G, n, L, Hkv):
    """Both take the exact codes as operands and the affine terms in 32 bits: the relative error
    against 64 bits is the verify kernel's. It is a norm over 150,000 to 400,000 outputs, most of it
    their bf16 rounding, so two draws of it agree to about 0.5 / sqrt(150,000) = 0.13%; K and V
    rounded to fp16 before the products show 3 to 5%. Scores with a standard deviation of 2."""
    from lagunalab_amd.q8_attn import _prefill_blocked, q8_prefill_attention
    rng = np.random.default_rng(G + n)
    kq, vq = (_buffers(dev, Q.randn_bf16(rng, (1, Hkv, n, 128)), n + 3) for _ in range(2))
    q = Q.round_bf16(2 * Q.randn_bf16(rng, (1, Hkv * G, L, 128)))
    qd = to_dev_bf16(q, dev)
    want = A.fused_attention(q, cache_np(kq), cache_np(vq), n, 128 ** -0.5, causal=True)

    def error(out):
        return np.linalg.norm(out.float().cpu().numpy() - want) / np.linalg.norm(want)
    got = error(q8_prefill_attention(qd, kq, vq, n, 128 ** -0.5))
    verify = error(_prefill_blocked(qd, kq, vq, n, 128 ** -0.5))
    assert got <= 1.01 * verify, (got, verify)


@pytest.mark.parametrize("G", [6, 3])
@pytest.mark.parametrize("n,L", [(500, 70), (3000, 70)], ids=["whole", "split"])
@pytest.mark.parametrize("kind", ["far keys", "large scores", "V groups", "V tiles"])
def test_prefill_operands_far_apart(dev, kind, n, L, G):
    """What the verify kernel serves and a dequantized fp16 operand does not hold: keys 2^36 times
    others of their tile (with scores far below theirs), scores of 2^30 and more, V groups of one
    head 2^-18 of each other, V sizes that jump by powers of two between regions of two 64-key tiles
    (at 500 keys in whole blocks: the exponent changes within one walk of the keys)."""
    from lagunalab_amd.q8_attn import q8_prefill_attention
    Hkv, cap = 2, n + 40
    assert _split(n, L, G, Hkv) == (n == 3000)
    rng = np.random.default_rng(n + G)
    q = Q.randn_bf16(rng, (1, Hkv, 1, 1, 128)) * np.float32(4.0)
    q = Q.round_bf16(q + 0.3 * Q.randn_bf16(rng, (1, Hkv, G, L, 128))).reshape(1, Hkv * G, L, 128)
    qdir = q[0, ::G, 0] / np.linalg.norm(q[0, ::G, 0], axis=-1, keepdims=True)
    k, v = (Q.randn_bf16(rng, (1, Hkv, n, 128)) for _ in range(2))
    if kind == "far keys":
        k[:, :, ::2] -= np.float32(2.0 ** 36) * qdir[None, :, None, :]
    elif kind == "large scores":
        k *= np.float32(2.0 ** 16)
        q = Q.round_bf16(Q.randn_bf16(rng, q.shape) * np.float32(2.0 ** 16))
    elif kind == "V groups":
        v[..., 64:] *= np.float32(2.0 ** -18)
    else:
        region = (np.arange(n) // 128) % 3
        k += np.where(region == 1, 6.0, -6.0).astype(np.float32)[:, None] * qdir[None, :, None, :]
        v *= (np.float32(2.0) ** np.array([4, -14, -5])[region]).astype(np.float32)[:, None]
    kq, vq = _buffers(dev, k, cap), _buffers(dev, v, cap)
    got = q8_prefill_attention(to_dev_bf16(q, dev), kq, vq, n, 128 ** -0.5).float().cpu().numpy()
    want = A.fused_attention(q, cache_np(kq), cache_np(vq), n, 128 ** -0.5, causal=True)
    assert np.isfinite(got).all()
    for g in (slice(0, 64), slice(64, 128)):
        # the parity bar, against each row's own largest value of the group
        mag = np.abs(want[..., g]).max(-1, keepdims=True)
        err = np.abs(got[..., g] - want[..., g])
        assert np.all(err <= 2e-3 * mag + RTOL * np.abs(want[..., g])), (kind, float((err / mag).max()))


@pytest.mark.parametrize("value", [float("nan"), float("inf")])
@pytest.mark.parametrize("word", ["K scale", "K bias", "V scale", "V bias"])
def test_prefill_infinity_in_a_key_reaches_the_rows_that_see_it(dev, word, value):
    """A NaN or infinity in one key of the chunk: the rows before it are what they are without it, the
    rows from it on are not finite. (A K scale or bias of -inf times a q sum can also give a score of
    -inf, a key without weight: rows with a NaN or a changed result both count as reached.)"""
    from lagunalab_amd.q8_attn import q8_prefill_attention
    rng = np.random.default_rng(9)
    n, L, G, Hkv, at = 700, 90, 6, 1, 650  # the chunk begins at key 610
    kq, vq = (_buffers(dev, Q.randn_bf16(rng, (1, Hkv, n, 128)), n) for _ in range(2))
    q = to_dev_bf16(Q.randn_bf16(rng, (1, Hkv * G, L, 128)), dev)
    clean = q8_prefill_attention(q, kq, vq, n, 128 ** -0.5).float()
    buf = (kq if word[0] == "K" else vq)[1 if word.endswith("scale") else 2]
    buf[0, 0, at, 0] = value
    got = q8_prefill_attention(q, kq, vq, n, 128 ** -0.5).float()
    i = at - (n - L)
    assert torch.allclose(got[:, :, :i], clean[:, :, :i], rtol=2.0 ** -7, atol=0)
    reached = ~torch.isclose(got[:, :, i:], clean[:, :, i:], rtol=2.0 ** -7, atol=0).all(-1)
    assert bool(reached.all())
    if value != value:
        assert bool(got[:, :, i:].isnan().any(-1).all())
