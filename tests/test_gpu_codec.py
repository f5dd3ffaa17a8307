"""GPU tests of the quantizer's and the dequantiser's launch shapes: whole and
partial workgroup runs (256 blocks; 1024 quads of values), destinations with
and without 16-byte alignment, FP32 and BF16 sources, rows from the middle of a
matrix.  Every byte and every value against the oracle, exactly."""
import numpy as np
import pytest

import oracle
import qwen3x_amd as q3x
from tests.helpers import Q4_0, Q8_0, random_blocks
from tests.test_gpu_parity import _torch, dev, host, say

pytestmark = pytest.mark.gpu


def _values(blocks):
    rng = np.random.default_rng(blocks)
    v = rng.normal(0, 0.02, (blocks, 32)).astype(np.float32)
    v = (v.view(np.uint32) & 0xffff0000).view(np.float32)  # exact in BF16, so both sources agree
    v[0, :] = 0.0
    if blocks > 2:
        v[1, 5] = v[1, 17] = -0.5  # the largest magnitude twice, once with either sign: the first wins
        v[1, 9] = 0.5
        v[2, 31] = 2.0
    return v


@pytest.mark.parametrize("type_", [Q8_0, Q4_0])
@pytest.mark.parametrize("offset", [0, 2, 7])
@pytest.mark.parametrize("blocks", [1, 3, 63, 256, 257, 1300])
def test_quantize_run_edges(type_, offset, blocks):
    torch = _torch()
    v = _values(blocks)
    want = oracle.quantize(type_, v)
    say(f"quantize type={type_} blocks={blocks} offset={offset}")
    for bf16 in (False, True):
        buf = torch.full((offset + want.size + 16,), 0xA5, dtype=torch.uint8, device="cuda:0")
        if bf16:
            q3x.quantize_bf16(type_, dev((v.view(np.uint32) >> 16).astype(np.uint16).view(np.int16)), blocks, 32,
                              buf[offset:])
        else:
            q3x.quantize(type_, dev(v), blocks, 32, buf[offset:])
        got = host(buf)
        assert np.array_equal(got[offset:offset + want.size], want)
        assert np.all(got[:offset] == 0xA5) and np.all(got[offset + want.size:] == 0xA5)


@pytest.mark.parametrize("type_", [Q8_0, Q4_0])
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("rows,cols", [(1, 32), (3, 96), (5, 4096), (4, 1024), (33, 160)])
def test_dequant_run_edges(type_, offset, rows, cols):
    torch = _torch()
    w = random_blocks(np.random.default_rng(rows * cols), type_, rows + 2, cols)
    want = oracle.dequant(w, type_, rows + 2, cols)[1:1 + rows]
    say(f"dequant type={type_} {rows}x{cols} offset={offset}")
    out = torch.full((offset + rows * cols + 4,), -7.0, dtype=torch.float32, device="cuda:0")
    q3x.dequant(q3x.Linear(dev(w), rows + 2, cols, type_), 1, rows, out[offset:])
    got = host(out)
    assert np.array_equal(got[offset:offset + rows * cols].reshape(rows, cols).view(np.uint32), want.view(np.uint32))
    assert np.all(got[:offset] == -7.0) and np.all(got[offset + rows * cols:] == -7.0)


@pytest.mark.parametrize("type_", [Q8_0, Q4_0])
@pytest.mark.parametrize("blocks", [1, 257])
def test_quantize_every_alignment(type_, blocks):
    """Destinations at every byte of a 16-byte word, a run shorter than one
    and runs of whole words between single bytes."""
    torch = _torch()
    v = _values(blocks)
    want = oracle.quantize(type_, v)
    src = dev(v)
    say(f"quantize type={type_} blocks={blocks} at offsets 0 to 16")
    for offset in range(17):
        buf = torch.full((offset + want.size + 16,), 0xA5, dtype=torch.uint8, device="cuda:0")
        q3x.quantize(type_, src, blocks, 32, buf[offset:])
        got = host(buf)
        assert np.array_equal(got[offset:offset + want.size], want)
        assert np.all(got[:offset] == 0xA5) and np.all(got[offset + want.size:] == 0xA5)
