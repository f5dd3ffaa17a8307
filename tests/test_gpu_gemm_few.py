"""GPU tests of the GEMM plans for 33 to 192 tokens (48 x 128, 80 x 256 and 96 x
256 tiles, 64 x 128 on two K halves over short K, up to 16 splits): token counts
at and past each tile's edge, ragged rows and K ranges, split over K and whole.
Against W x in float64 within the bound of the GEMM tests (1e-5 ||w|| ||x||),
the split launch against the whole one, twice bit for bit, and accumulating; a
workspace sized for more tokens; and an engine's prompts, whose paired gate and
up launch is too small for those tiles (test_gpu_gemm_plans.py runs it on them)."""
import numpy as np
import pytest

import qwen3x_amd as q3x
from tests.engine_models import CONFIGS, synthetic_model
from tests.helpers import Q4_0, Q8_0, dequant_numpy, random_blocks
from tests.test_gpu_parity import _torch, bits, dev, host, say

pytestmark = pytest.mark.gpu

TILES = {48: 128, 64: 128, 80: 256, 96: 256, 128: 256}


# The tile height that each count is to take on these matrices.
FEW = [(33, 48), (48, 48), (49, 64), (64, 64), (65, 80), (80, 80), (81, 96), (96, 96), (129, 80), (160, 80)]


@pytest.mark.parametrize("type_", [Q8_0, Q4_0])
@pytest.mark.parametrize("rows,cols,count,height",
                         [(rows, cols, *few) for rows, cols in [(8300, 4128), (4097, 6144)] for few in FEW] +
                         [(4097, 6144, 97, 128), (4097, 6144, 128, 128), (4097, 6144, 161, 96), (4097, 6144, 192, 96),
                          (8300, 4128, 161, 64), (8300, 4128, 192, 64)])
def test_few_token_tiles(type_, rows, cols, count, height):
    torch = _torch()
    rng = np.random.default_rng(rows + cols + count + type_)
    w = random_blocks(rng, type_, rows, cols)
    X = rng.normal(0, 1, (count, cols)).astype(np.float32)
    wd = dequant_numpy(w, type_, rows, cols).astype(np.float32)
    Xd = dev(X)
    want = host(Xd.double() @ dev(wd).double().T)
    bound = 1e-5 * np.linalg.norm(X.astype(np.float64), axis=1)[:, None] * np.linalg.norm(wd, axis=1)[None, :]
    lin = q3x.Linear(dev(w), rows, cols, type_)
    nbytes = q3x.gemm_workspace_bytes(lin, count)
    unit = -(-rows // TILES[height]) * -(-count // height) * height * TILES[height] * 4
    say(f"few-token tiles type={type_} {rows}x{cols} count={count} splits={nbytes / unit:g}")
    assert nbytes % unit == 0 and nbytes > 0, "the plan must take this tile"
    ws = torch.empty(max(nbytes, 16), dtype=torch.uint8, device="cuda:0")
    Y, Y2 = (torch.full((count * rows + 8,), 3.0, dtype=torch.float32, device="cuda:0") for _ in range(2))
    q3x.batch_mv_ws(lin, Xd, Y, count, ws)
    got = host(Y)
    assert np.all(got[count * rows:] == 3.0), "wrote past the output"
    got = got[:count * rows].reshape(count, rows)
    assert np.all(np.abs(got - want) <= bound)
    q3x.batch_mv(lin, Xd, Y2, count)  # no workspace: a whole launch
    whole = host(Y2)
    assert np.all(whole[count * rows:] == 3.0), "wrote past the output"
    assert np.all(np.abs(whole[:count * rows].reshape(count, rows) - want) <= bound)
    q3x.batch_mv_ws(lin, Xd, Y2, count, ws)
    assert np.array_equal(bits(host(Y2)), bits(host(Y)))
    q3x.batch_mv_ws(lin, Xd, Y2, count, ws, add=True)  # the same sums again, added: exactly twice
    assert np.array_equal(bits(host(Y2)[:count * rows]), bits((got + got).reshape(-1)))


@pytest.mark.parametrize("type_", [Q8_0, Q4_0])
@pytest.mark.parametrize("rows,cols,most,counts", [(12288, 4096, 192, (40, 64, 80, 96, 128)), (4096, 12288, 192, (96, 128)),
                                                   (17408, 5120, 512, (176, 256))])
def test_workspace_sized_for_more_tokens(type_, rows, cols, most, counts):
    """The workspace of a larger count keeps the split: the bits of a call with
    the count's own, and not those of the unsplit launch."""
    torch = _torch()
    rng = np.random.default_rng(rows + type_)
    lin = q3x.Linear(dev(random_blocks(rng, type_, rows, cols)), rows, cols, type_)
    shared = torch.empty(q3x.gemm_workspace_bytes(lin, most), dtype=torch.uint8, device="cuda:0")
    for count in counts:
        say(f"workspace of {most} tokens type={type_} {rows}x{cols} count={count}")
        X = dev(rng.normal(0, 1, (count, cols)).astype(np.float32))
        own = torch.empty(q3x.gemm_workspace_bytes(lin, count), dtype=torch.uint8, device="cuda:0")
        Y = [torch.full((count, rows), 3.0, dtype=torch.float32, device="cuda:0") for _ in range(3)]
        q3x.batch_mv_ws(lin, X, Y[0], count, shared)
        q3x.batch_mv_ws(lin, X, Y[1], count, own)
        q3x.batch_mv(lin, X, Y[2], count)
        assert torch.equal(Y[0].view(torch.int32), Y[1].view(torch.int32))
        assert not torch.equal(Y[0].view(torch.int32), Y[2].view(torch.int32))


@pytest.mark.parametrize("type_", [Q8_0, Q4_0])
def test_engine_prompts_against_single_tokens(type_):
    """Prompts' GEMMs (the paired gate and up launch among them) against the
    same tokens one by one, each within the engine tests' bound of the
    reference forward, so within twice that of each other."""
    _torch()
    fields = dict(CONFIGS["dense_q8"], matrix_type=type_, H=1024, I=4096, VH=8, KH=2, AH=4)
    config, image, _ = synthetic_model(fields, seed=60 + type_)
    tokens = np.random.default_rng(type_).integers(0, fields["V"], 160).astype(np.int32)
    weights = dev(image)
    with q3x.Engine(config, weights, context=len(tokens)) as engine:
        want = []
        for i in range(len(tokens)):
            engine.forward(tokens[i:i + 1])
            want.append(engine.logits())
        for prompt in (40, 64, 77, 90, 128, 160):
            say(f"engine type={type_}: prompt {prompt}")
            engine.reset()
            engine.forward(tokens[:prompt])
            assert np.all(np.abs(engine.logits() - want[prompt - 1]) <= 2 * (2e-4 + 2e-4 * np.abs(want[prompt - 1])))
