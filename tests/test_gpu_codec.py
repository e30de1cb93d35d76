"""NF4 codec on the GPU vs the CPU oracle: codes, absmax, nested statistics,
resolved scales and dequantised bf16/fp32 weights must be bit-exact."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import nf4_oracle as O
from tests._util import np_bits, np_f32, oracle_weight, seeded

import molt_amd
from molt_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,block", [((64, 64), 64), ((70, 65), 64), ((8, 8), 16), ((33, 7), 32),
                                         ((128, 96), 64), ((5, 200), 50)])
@pytest.mark.parametrize("order", [0, 1])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_quantize_codes_and_absmax_bit_exact(shape, block, order, dtype):
    print(f"quantize shape={shape} block={block} order={order} dtype={dtype}", flush=True)
    x = seeded(shape, 100 + block + order, std=0.02, dtype=dtype)
    packed, absmax = ops.nf4_quantize(x, block, order, molt_amd.NF4_CODEBOOK.cuda())
    idx, am = O.quantize_blocks(np_f32(x), block)
    assert np.array_equal(np_f32(absmax).view(np.uint32), am.view(np.uint32))
    assert np.array_equal(packed.cpu().numpy(), O.pack_nibbles(idx, order))


@pytest.mark.parametrize("block", [32, 64])
def test_quantize_special_values(block):
    """Zero blocks (absmax clamped to FLT_MIN), exact codes, ties; block 64
    takes the one-element-per-lane path, block 32 the pair-per-lane one."""
    code = O.NF4_CODE
    lo, hi = code[9], code[10]
    mid = np.float32((np.float64(lo) + np.float64(hi)) / 2)
    x = np.concatenate([np.zeros(64, np.float32), code * np.float32(3.0), code * np.float32(-0.25),
                        np.array([1.0, mid, -mid] + [0.0] * 29, np.float32)]).astype(np.float32)
    xt = torch.from_numpy(x).cuda()
    for order in (0, 1):
        packed, absmax = ops.nf4_quantize(xt, block, order, molt_amd.NF4_CODEBOOK.cuda())
        idx, am = O.quantize_blocks(x, block)
        assert np.array_equal(np_f32(absmax).view(np.uint32), am.view(np.uint32))
        assert np.array_equal(packed.cpu().numpy(), O.pack_nibbles(idx, order))


def test_quantize_block64_more_blocks_than_one_pass():
    """135,168 blocks of 64: more than one pass of the block-64 path's grid
    (2048 workgroups x 4 waves x 2 units of 8 blocks), the second pass partial."""
    shape = (4096, 2112)
    print(f"quantize block64 multi-pass shape={shape}", flush=True)
    x = seeded(shape, 7, std=0.02, dtype=torch.bfloat16)
    packed, absmax = ops.nf4_quantize(x, 64, 1, molt_amd.NF4_CODEBOOK.cuda())
    idx, am = O.quantize_blocks(np_f32(x), 64)
    assert np.array_equal(np_f32(absmax).view(np.uint32), am.view(np.uint32))
    assert np.array_equal(packed.cpu().numpy(), O.pack_nibbles(idx, 1))


@pytest.mark.parametrize("n", [1, 255, 256, 4096, 4097, 70000, 300000])
def test_double_quantize_bit_exact(n):
    print(f"double quantize n={n}", flush=True)
    g = torch.Generator().manual_seed(n)
    absmax = (torch.randn(n, generator=g).abs() * 0.02 + 1e-4).float()
    code2 = molt_amd.dynamic_map()
    q, absmax2, offset = ops.nf4_double_quantize(absmax.cuda(), code2.cuda(), 256)
    oq, oa2, ooff, _ = O.double_quantize(absmax.numpy(), code2.numpy())
    assert np.float32(offset.item()).view(np.uint32) == np.float32(ooff).view(np.uint32)
    assert np.array_equal(np_f32(absmax2).view(np.uint32), oa2.view(np.uint32))
    assert np.array_equal(q.cpu().numpy(), oq)


@pytest.mark.parametrize("shape", [(64, 64), (70, 65), (256, 384), (4864, 896)])
@pytest.mark.parametrize("nested", [True, False])
def test_quantize_4bit_dequantize_4bit_bit_exact(shape, nested):
    print(f"quantize_4bit/dequantize_4bit shape={shape} nested={nested}", flush=True)
    w = seeded(shape, 7, std=0.02, dtype=torch.float32)
    packed, qs = molt_amd.quantize_4bit(w, blocksize=64, compress_statistics=nested)
    ow = O.quantize_bnb_layout(np_f32(w), 64, nested=nested)
    assert np.array_equal(packed.reshape(-1).cpu().numpy(), ow.packed[: packed.numel()])
    if nested:
        assert np.array_equal(qs.absmax.cpu().numpy(), ow.q)
        assert np.float32(float(qs.offset)).view(np.uint32) == np.float32(ow.offset).view(np.uint32)
    scales = molt_amd.resolved_nf4_scales(qs)
    assert np.array_equal(np_f32(scales).view(np.uint32), ow.scales.view(np.uint32))
    dense = molt_amd.dequantize_4bit(packed, qs)
    assert dense.dtype == torch.float32 and dense.shape == shape
    assert np.array_equal(np_f32(dense).view(np.uint32), ow.dequant_f32().view(np.uint32))
    dense_bf16 = molt_amd.dequantize_4bit(packed, qs, torch.bfloat16)
    assert np.array_equal(np_bits(dense_bf16), ow.dequant_bf16_bits())


def test_dequantize_bf16_weights_of_bf16_input():
    w = seeded((1536, 256), 944, std=1.0, dtype=torch.bfloat16)
    packed, qs = molt_amd.quantize_4bit(w, blocksize=64, compress_statistics=True)
    assert qs.dtype == torch.bfloat16
    ow = oracle_weight(packed, qs)
    assert np.array_equal(np_bits(molt_amd.dequantize_4bit(packed, qs)), ow.dequant_bf16_bits())


def test_cleanroom_nf4tensor_round_trip():
    """streaming/nf4.py semantics: low nibble first, fp32 scales, padding."""
    torch.manual_seed(1)
    value = torch.randn(64, 64)
    t = molt_amd.NF4Tensor.quantize(value, block_size=64)
    ow = O.quantize_cleanroom(value.numpy(), 64)
    assert np.array_equal(t.packed.numpy(), ow.packed)
    assert np.array_equal(t.scales.numpy().view(np.uint32), ow.scales.view(np.uint32))
    assert t.storage_bytes == value.numel() // 2 + value.numel() // 64 * 4
    restored = t.dequantize(device="cuda").cpu()
    assert np.array_equal(restored.numpy().view(np.uint32), ow.dequant_f32().view(np.uint32))
    assert torch.mean((restored - value) ** 2).sqrt() < 0.15
    odd = torch.randn(3, 37)
    t2 = molt_amd.NF4Tensor.quantize(odd, block_size=16)
    ow2 = O.quantize_cleanroom(odd.numpy(), 16)
    assert np.array_equal(t2.packed.numpy(), ow2.packed)
    bf = t2.dequantize(device="cuda", dtype=torch.bfloat16).cpu()
    assert np.array_equal(np_bits(bf), ow2.dequant_bf16_bits())


_TABLES = {
    "nf4": O.NF4_CODE,
    "reversed": O.NF4_CODE[::-1].copy(),                     # not sorted: the definition's scan
    "close": np.sort(np.concatenate([O.NF4_CODE[:14], O.NF4_CODE[9:10] + 2e-4, O.NF4_CODE[3:4] - 0.004])),
    "uneven": np.linspace(-0.9, 1.0, 16).astype(np.float32) ** 3,   # thresholds closer than a bucket
}


@pytest.mark.parametrize("table", list(_TABLES))
@pytest.mark.parametrize("n", [2, 64, 65, 64 * 7 + 6, 64 * 8, 64 * 9 + 62, 64 * 8 * 4 * 3 + 34])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_quantize_block64_against_the_scan(n, dtype, table):
    """Few blocks of 64 (a wave to a block) at the edges of a wave's and a pass's blocks, for each kind of table, from
    aligned and unaligned inputs: every code and absmax as the definition's scan."""
    print(f"quantize block64 n={n} dtype={dtype} table={table}", flush=True)
    code = _TABLES[table]
    x = seeded((n + 1,), 900 + n, std=0.02, dtype=dtype)
    for src in (x[:n].clone(), x[1:]):
        packed, absmax = ops.nf4_quantize(src, 64, 1, torch.from_numpy(code).cuda())
        idx, am = O.quantize_blocks(np_f32(src), 64, code)
        assert np.array_equal(np_f32(absmax).view(np.uint32), am.view(np.uint32))
        assert np.array_equal(packed.cpu().numpy(), O.pack_nibbles(idx, 1))


def test_quantize_block64_at_the_thresholds_and_out_of_range_blocks():
    """The floats around every midpoint under absmax 1 and under odd absmax values, and blocks whose absmax (zero,
    denormal, tiny, huge, infinite) leaves the reciprocal's range."""
    mids = (O.NF4_CODE[:-1].astype(np.float64) + O.NF4_CODE[1:]) / 2
    rows = []
    for am in (1.0, 0.0213, 3.7e-3, 1.999999, 2.0 ** -59, 2.0 ** 59, 2.0 ** -61, 2.0 ** 61, 1e-38, 3e38):
        for step in range(-4, 5):
            near = (mids * am).astype(np.float32)
            for _ in range(abs(step)):
                near = np.nextafter(near, np.float32(np.inf if step > 0 else -np.inf))
            rows.append(np.concatenate([near, -near, [np.float32(am)], np.zeros(33, np.float32)]))
    rows += [np.zeros(64), np.full(64, 1e-45), np.r_[np.inf, np.zeros(62), 1.0]]
    x = np.stack(rows).astype(np.float32)
    packed, absmax = ops.nf4_quantize(torch.from_numpy(x).cuda(), 64, 0, molt_amd.NF4_CODEBOOK.cuda())
    with np.errstate(invalid="ignore"):
        idx, am = O.quantize_blocks(x, 64)
    assert np.array_equal(np_f32(absmax).view(np.uint32), am.view(np.uint32))
    assert np.array_equal(packed.cpu().numpy(), O.pack_nibbles(idx, 0))


def _table_blocks():
    """Blocks of 64 from which the quantiser looks its codes up (below, it scans them): 40 per CU."""
    return 40 * torch.cuda.get_device_properties(0).multi_processor_count


@pytest.mark.parametrize("table", list(_TABLES))
@pytest.mark.parametrize("extra", [-64, -63, 0, 64 * 8 * 4 * 3 + 34])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_quantize_block64_around_the_table_line(extra, dtype, table):
    """Just below, at and above the number of blocks where the quantiser goes from the scan to the threshold table,
    with whole and ragged last blocks, aligned and unaligned inputs and every kind of table."""
    n = _table_blocks() * 64 + extra
    print(f"quantize block64 n={n} dtype={dtype} table={table}", flush=True)
    code = _TABLES[table]
    x = seeded((n + 1,), 950 + extra % 7, std=0.02, dtype=dtype)
    for src in (x[:n].clone(), x[1:]):
        packed, absmax = ops.nf4_quantize(src, 64, 1, torch.from_numpy(code).cuda())
        idx, am = O.quantize_blocks(np_f32(src), 64, code)
        assert np.array_equal(np_f32(absmax).view(np.uint32), am.view(np.uint32))
        assert np.array_equal(packed.cpu().numpy(), O.pack_nibbles(idx, 1))


def test_quantize_block64_thresholds_through_the_table():
    """The floats around every midpoint, and blocks out of the reciprocal's range, in a weight large enough for the
    threshold table; eight equal blocks in a row, so that whole waves of blocks are in range and take it."""
    mids = (O.NF4_CODE[:-1].astype(np.float64) + O.NF4_CODE[1:]) / 2
    rows = []
    for am in (1.0, 0.0213, 3.7e-3, 1.999999, 2.0 ** -59, 2.0 ** 59, 2.0 ** -61, 2.0 ** 61, 1e-38, 3e38):
        for step in range(-4, 5):
            near = (mids * am).astype(np.float32)
            for _ in range(abs(step)):
                near = np.nextafter(near, np.float32(np.inf if step > 0 else -np.inf))
            rows.append(np.concatenate([near, -near, [np.float32(am)], np.zeros(33, np.float32)]))
    rows += [np.zeros(64), np.full(64, 1e-45), np.r_[np.inf, np.zeros(62), 1.0]]
    x = np.repeat(np.stack(rows).astype(np.float32), 8, axis=0)
    times = -(-_table_blocks() // len(x))
    packed, absmax = ops.nf4_quantize(torch.from_numpy(np.tile(x, (times, 1))).cuda(), 64, 0,
                                      molt_amd.NF4_CODEBOOK.cuda())
    with np.errstate(invalid="ignore"):
        idx, am = O.quantize_blocks(x, 64)
    assert np.array_equal(np_f32(absmax).view(np.uint32), np.tile(am.reshape(-1), times).view(np.uint32))
    assert np.array_equal(packed.cpu().numpy().reshape(times, -1), np.tile(O.pack_nibbles(idx, 0).reshape(1, -1), (times, 1)))


@pytest.mark.parametrize("table", ["dynamic", "ties", "unsorted"])
def test_double_quantize_tables(table):
    """Sorted tables (with equal entries: the first index wins) take the search, an unsorted one the scan."""
    code2 = molt_amd.dynamic_map()
    if table == "ties":
        code2 = torch.sort((code2 * 40).round() / 40).values
    elif table == "unsorted":
        code2 = code2[torch.randperm(256, generator=torch.Generator().manual_seed(3))]
    g = torch.Generator().manual_seed(5)
    absmax = (torch.randn(5000, generator=g).abs() * 0.02 + 1e-4).float()
    q, absmax2, offset = ops.nf4_double_quantize(absmax.cuda(), code2.cuda(), 256)
    oq, oa2, ooff, _ = O.double_quantize(absmax.numpy(), code2.numpy())
    assert np.array_equal(np_f32(absmax2).view(np.uint32), oa2.view(np.uint32))
    assert np.array_equal(q.cpu().numpy(), oq)
