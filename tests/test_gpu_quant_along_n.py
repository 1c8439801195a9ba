"""The fused quantizer with blocks along N, both 16-bit types, at what its loads, its reduction across the lanes and its
rule for zeros have to get right: columns that end inside a tile, strided and unaligned sources, extreme values, and
weights that are no numbers.  Bit for bit against the oracle (reference: src/mickey/blk_q4/f16_quant_sm80.cuh:96-141,
225-315), through the C ABI."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

TYPES = pytest.mark.parametrize("bf16", [False, True], ids=["fp16", "bf16"])
OFFSETS = pytest.mark.parametrize("has_offsets", [True, False])
BLOCKS = pytest.mark.parametrize("bs", [16, 32, 64])


def to_bits(oracle, values, bf16):
    return oracle.f32_to_bf16(values.astype(np.float32)) if bf16 else values.astype(np.float16).view(np.uint16)


def check(oracle, capi, device, bs, bits, has_offsets, bf16, ld=None, shift=0):
    """quantizes the [N, K] bit patterns, laid out with leading dimension ld from element `shift` of an aligned buffer"""
    n, k = bits.shape
    ld = k if ld is None else ld
    dtype = torch.bfloat16 if bf16 else torch.float16
    buf = np.full(shift + n * ld, 0x3c00, np.uint16)
    buf[shift:].reshape(n, ld)[:, :k] = bits
    src = torch.from_numpy(buf.view(np.int16)).to(device).view(dtype)[shift:]
    w_elems, meta_elems = capi.quant_size(bs, False, k, n)
    q_w = torch.full((w_elems,), 0xA5, dtype=torch.uint8, device=device)
    q_s = torch.full((meta_elems,), float("nan"), dtype=dtype, device=device)
    q_zp = torch.full((meta_elems,), 0xEE, dtype=torch.uint8, device=device) if has_offsets else None
    capi.quant(bs, False, src, q_w, q_s, q_zp, rows=k, columns=n, ld=ld, bf16=bf16)
    torch.cuda.synchronize()
    canon, s, z = oracle.quantize(bs, False, bits if bf16 else bits.view(np.float16), has_offsets, bf16=bf16)
    # a weight that is infinite or no number becomes the nibble 0 (the oracle's conversion of it is not defined)
    finite = (bits & (0x7f80 if bf16 else 0x7c00)) != (0x7f80 if bf16 else 0x7c00)
    canon = oracle.canonical_from_nibbles(np.where(finite, oracle.nibbles_from_canonical(canon), 0).astype(np.uint8))
    ps, pz = oracle.prepack_meta_sm80(bs, False, k, n, s, z)
    assert np.array_equal(q_s.view(torch.int16).cpu().numpy().view(np.uint16), ps.view(np.uint16)), "scales differ"
    if has_offsets:
        assert np.array_equal(q_zp.cpu().numpy(), pz), "zero-points differ"
    assert np.array_equal(q_w.cpu().numpy(), oracle.native_from_canonical(canon)), "packed weights differ"


def gaussian(seed, n, k):
    return np.random.default_rng(seed).standard_normal((n, k)) * 0.02


@TYPES
@OFFSETS
@pytest.mark.parametrize("bs,rows,columns", [(16, 64, 32), (16, 320, 96), (32, 576, 160), (64, 192, 64), (64, 320, 192)])
def test_columns_that_end_inside_a_tile(oracle, capi, device, bs, has_offsets, rows, columns, bf16):
    w = gaussian(bs + rows + columns, columns, rows)
    w[:, 5] = -0.0
    w[0, 9], w[1:, 9] = -0.0, 0.0   # an all-zero block's scale takes the sign of its first weight
    check(oracle, capi, device, bs, to_bits(oracle, w, bf16), has_offsets, bf16)


@TYPES
@BLOCKS
@pytest.mark.parametrize("pad,shift", [(8, 0), (3, 0), (0, 1), (5, 3)])
def test_strided_and_unaligned_source(oracle, capi, device, bs, pad, shift, bf16):
    rows, columns = 192, 192
    bits = to_bits(oracle, gaussian(bs + pad + shift, columns, rows), bf16)
    for has_offsets in (True, False):
        check(oracle, capi, device, bs, bits, has_offsets, bf16, ld=rows + pad, shift=shift)


@TYPES
@OFFSETS
@BLOCKS
def test_extreme_values(oracle, capi, device, bs, has_offsets, bf16):
    """constant blocks, ties between the two extremes, large, tiny and subnormal (fp16) magnitudes, zeros of both signs"""
    rng = np.random.default_rng(99)
    w = gaussian(98, 192, 256)
    w[:64, 0] = 0.0
    w[:64, 1] = -0.0
    w[:64, 2], w[5, 2] = 0.0, -0.0
    w[:64, 3], w[0, 3] = 0.0, -0.0
    w[64:128, 4] = 3.0
    w[64:128, 5] = -3.0
    w[:64, 6] = rng.standard_normal(64) * 3000
    w[:64, 7] = rng.standard_normal(64) * 1e-6
    w[:64, 8], w[3, 8] = 65504.0, -65504.0
    w[:64, 9], w[3, 9] = -65504.0, 65504.0
    w[64:128, 255] = 6e-8
    check(oracle, capi, device, bs, to_bits(oracle, w, bf16), has_offsets, bf16)


@BLOCKS
@pytest.mark.parametrize("kind,has_offsets,bf16", [
    ("quiet", True, False), ("quiet", False, False), ("signalling", True, False), ("signalling", False, False),
    ("infinite", False, False), ("quiet", True, True), ("quiet", False, True), ("infinite", False, True)])
def test_weights_that_are_no_numbers(oracle, capi, device, bs, kind, has_offsets, bf16):
    """a NaN counts in no minimum and no maximum (in bf16 that holds for quiet ones); an infinite extreme makes an infinite
    scale (without zero-points; with them the scale is a difference of the extremes, and not defined)"""
    bits = to_bits(oracle, gaussian(97, 192, 320), bf16)
    infinite = 0x7f80 if bf16 else 0x7c00
    value = {"quiet": infinite | (0x40 if bf16 else 0x200), "signalling": infinite | 1, "infinite": infinite}[kind]
    for k in range(320):   # one per block of a k at most, at every place of a block in turn, of both signs
        bits[(7 * k) % bs + bs * (k % (192 // bs)), k] = value | (0x8000 if k % 3 == 0 else 0)
    check(oracle, capi, device, bs, bits, has_offsets, bf16)


@TYPES
@BLOCKS
@pytest.mark.parametrize("signalling", [False, True])
def test_blocks_without_any_number_scale_by_their_first_weight(capi, device, bs, signalling, bf16):
    """without zero-points: the scale is the first weight's NaN, made quiet, with its sign and payload"""
    n, k = 192, 320
    infinite, quiet = (0x7f80, 0x40) if bf16 else (0x7c00, 0x200)
    rng = np.random.default_rng(bs)
    bits = (infinite | (0 if signalling else quiet) | rng.integers(1, quiet, (n, k)) | (rng.integers(0, 2, (n, k)) << 15)).astype(np.uint16)
    dtype = torch.bfloat16 if bf16 else torch.float16
    w_elems, meta_elems = capi.quant_size(bs, False, k, n)
    q_w = torch.full((w_elems,), 0xA5, dtype=torch.uint8, device=device)
    q_s = torch.zeros(meta_elems, dtype=dtype, device=device)
    capi.quant(bs, False, torch.from_numpy(bits.view(np.int16)).to(device).view(dtype), q_w, q_s, None, bf16=bf16)
    torch.cuda.synchronize()
    # packed order of the scales: inside 16 rows, rows 2t, 2t + 1, 2t + 8, 2t + 9 at 4t .. 4t + 3
    order = [r for t in range(4) for r in (2 * t, 2 * t + 1, 2 * t + 8, 2 * t + 9)]
    want = (bits[::bs] | quiet).reshape(n // bs, k // 16, 16)[:, :, order].reshape(-1)
    assert np.array_equal(q_s.view(torch.int16).cpu().numpy().view(np.uint16), want)
    assert not q_w.cpu().numpy().any()   # a weight that is no number becomes the nibble 0
