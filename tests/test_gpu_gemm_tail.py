"""GPU tests of the GEMM launches that split only the tiles of their last,
short round over K: token and row counts some tiles past the CU count, ragged
on both edges and over K.  Against W x in float64 within the bound of the
GEMM tests (1e-5 ||w|| ||x||), against the unsplit launch, twice bit for bit,
and accumulating."""
import numpy as np
import pytest

import qwen3x_amd as q3x
from tests import test_gpu_moe_layer as layers
from tests.helpers import Q4_0, Q8_0, dequant_numpy, random_blocks
from tests.test_gpu_parity import _torch, bits, dev, host, say

pytestmark = pytest.mark.gpu

CUS = 256
TILE = 128 * 256 * 4  # bytes of a unit's sums


@pytest.mark.parametrize("type_", [Q8_0, Q4_0])
@pytest.mark.parametrize("rows,cols,count", [(16640, 1024, 512), (17300, 1056, 500), (8400, 1056, 900)])
def test_gemm_tail_split(type_, rows, cols, count):
    torch = _torch()
    rng = np.random.default_rng(rows + cols + count + type_)
    w = random_blocks(rng, type_, rows, cols)
    X = rng.normal(0, 1, (count, cols)).astype(np.float32)
    wd = dequant_numpy(w, type_, rows, cols).astype(np.float64)
    want = X.astype(np.float64) @ wd.T
    bound = 1e-5 * np.linalg.norm(X.astype(np.float64), axis=1)[:, None] * np.linalg.norm(wd, axis=1)[None, :]
    lin = q3x.Linear(dev(w), rows, cols, type_)
    nbytes = q3x.gemm_workspace_bytes(lin, count)
    tail = -(-rows // 256) * -(-count // 128) - CUS
    assert nbytes > 0 and nbytes % (TILE * tail) == 0, "the plan must split the last round's tiles"
    say(f"gemm tail split type={type_} {rows}x{cols} count={count} tail={tail} units={nbytes // TILE}")
    ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda:0")
    Xd = dev(X)
    Y, Y2 = (torch.full((count, rows), float("nan"), dtype=torch.float32, device="cuda:0") for _ in range(2))
    q3x.batch_mv_ws(lin, Xd, Y, count, ws)
    got = host(Y)
    assert np.all(np.abs(got - want) <= bound)
    q3x.batch_mv(lin, Xd, Y2, count)
    assert np.all(np.abs(got - host(Y2)) <= bound)
    q3x.batch_mv_ws(lin, Xd, Y2, count, ws)
    assert np.array_equal(bits(host(Y2)), bits(got))
    q3x.batch_mv_ws(lin, Xd, Y2, count, ws, add=True)  # the same sums again, added: exactly twice
    assert np.array_equal(bits(host(Y2)), bits(got + got))


# The paired gate and up launch: a shared expert of 2 x 8320 rows over 500
# tokens is 260 tiles of 128 x 256, 4 past the CUs.  (test_gpu_gemm_plans.py
# asserts such a plan for this launch and the tails of the other tiles.)
def test_paired_tail_split():
    layers.test_moe_layer_parity(Q8_0, 2, 1024, 8448, 8320, 1, 500)
