"""GPU tests of the few-token GEMM (at most 32 tokens): every tile height and
its edges, row counts around the 16-row tiles and around the row tiles per
workgroup, rows shorter than the waves' K units, both formats.  Each output
against W x in float64 within the bound of the GEMM tests (1e-5 ||w|| ||x||),
and against the general tiles (reached through a matrix that is not 16-byte
aligned) within the two paths' FP32 rounding."""
import numpy as np
import pytest

import oracle
import qwen3x_amd as q3x
from tests.helpers import Q4_0, Q8_0, dequant_numpy, random_blocks, row_bound
from tests import test_gpu_moe_layer as layers
from tests.test_gpu_parity import _torch, dev, host, moe_bound, say

pytestmark = pytest.mark.gpu


def _run(type_, w, rows, cols, X, offset, add):
    torch = _torch()
    buf = torch.zeros(offset + w.size + 64, dtype=torch.uint8, device="cuda:0")
    buf[offset:offset + w.size] = dev(w.reshape(-1))
    T = X.shape[0]
    out = torch.full((T * rows + 8,), 3.0, dtype=torch.float32, device="cuda:0")
    q3x.batch_mv(q3x.Linear(buf[offset:offset + w.size], rows, cols, type_), dev(X), out, T, add=add)
    got = host(out)
    assert np.all(got[T * rows:] == 3.0), "wrote past the output"
    return got[:T * rows].reshape(T, rows).astype(np.float64) - (3.0 if add else 0.0)


@pytest.mark.parametrize("type_", [Q8_0, Q4_0])
@pytest.mark.parametrize("tokens", [1, 4, 5, 8, 9, 16, 17, 32, 33])
@pytest.mark.parametrize("rows,cols", [(1, 256), (15, 512), (49, 2304), (33, 4096), (4097, 1024), (8200, 256),
                                       (12300, 256), (1, 32), (33, 32), (17, 96), (31, 160), (100, 288), (3, 1056),
                                       (47, 4128), (18, 4160), (8200, 96)])
def test_few_token_gemm(type_, tokens, rows, cols):
    rng = np.random.default_rng(type_ + tokens * 64 + rows)
    w = random_blocks(rng, type_, rows, cols)
    X = rng.normal(0, 1, (tokens, cols)).astype(np.float32)
    wd = dequant_numpy(w, type_, rows, cols).astype(np.float64)
    want = X.astype(np.float64) @ wd.T
    bound = np.stack([row_bound(wd, x) for x in X])
    say(f"few-token gemm type={type_} {tokens}x{rows}x{cols}")
    got = _run(type_, w, rows, cols, X, 0, False)
    assert np.all(np.abs(got - want) <= bound)
    # Reading 3 back after adding costs up to half an ulp of the sum.
    added = _run(type_, w, rows, cols, X, 0, True)
    assert np.all(np.abs(added - want) <= bound + 2.0 ** -23 * (3.0 + np.abs(want)))
    dword = _run(type_, w, rows, cols, X, 4, False)  # a matrix aligned to 4 bytes only
    assert np.all(np.abs(dword - want) <= bound)
    general = _run(type_, w, rows, cols, X, 2, False)
    # Two FP32 sums of the same exact products: at most 2 (K + 40) 2^-24 of
    # the sum of their magnitudes, far below the bound above.
    scale = np.abs(X).astype(np.float64) @ np.abs(wd).T
    assert np.all(np.abs(got - general) <= 2 * (cols + 40) * 2.0 ** -24 * scale)


@pytest.mark.parametrize("type_", [Q8_0, Q4_0])
@pytest.mark.parametrize("tokens", [3, 7, 16])
def test_few_token_gemm_keeps_tokens_apart(type_, tokens):
    """An infinite activation reaches its own token's outputs only, in every
    row group that shares operand registers."""
    rows, cols = 64, 1024
    rng = np.random.default_rng(tokens)
    w = random_blocks(rng, type_, rows, cols)
    X = rng.normal(0, 1, (tokens, cols)).astype(np.float32)
    clean = _run(type_, w, rows, cols, X, 0, False)
    for col in (0, 33, 64, 100, 1023):
        bad = X.copy()
        bad[1, col] = np.inf
        got = _run(type_, w, rows, cols, bad, 0, False)
        keep = [t for t in range(tokens) if t != 1]
        assert np.array_equal(got[keep], clean[keep])
        assert not np.isfinite(got[1]).all()


@pytest.mark.parametrize("type_", [Q8_0, Q4_0])
@pytest.mark.parametrize("cols", [96, 1056, 4128])
def test_few_token_gemm_keeps_tokens_apart_at_the_row_end(type_, cols):
    """The same where K ends in a short unit: its registers also hold the next
    row's first blocks and the last block's activations again."""
    rows, tokens = 47, 7
    rng = np.random.default_rng(cols)
    w = random_blocks(rng, type_, rows, cols)
    X = rng.normal(0, 1, (tokens, cols)).astype(np.float32)
    clean = _run(type_, w, rows, cols, X, 0, False)
    for col in (0, cols - 33, cols - 32, cols - 1):
        bad = X.copy()
        bad[1, col] = np.inf
        got = _run(type_, w, rows, cols, bad, 0, False)
        keep = [t for t in range(tokens) if t != 1]
        assert np.array_equal(got[keep], clean[keep])
        assert not np.isfinite(got[1]).any()


@pytest.mark.parametrize("type_", [Q8_0, Q4_0])
@pytest.mark.parametrize("E,k,tokens", [(16, 2, 2), (16, 2, 4), (8, 2, 12), (4, 2, 20), (4, 2, 40), (300, 1, 5)])
@pytest.mark.parametrize("H,I", [(256, 256), (288, 96), (320, 160), (1056, 32)])
def test_few_pair_experts(type_, E, k, tokens, H, I):
    """The routed experts where an expert gets few pairs: every tile height
    (4, 8, 16, 32 pairs), spread and skewed routing (one expert holding every
    token: many tiles of it), ids out of range, rows of any block count.
    Against the oracle, and against the 80-pair tiles (reached through pools
    that are not dword aligned)."""
    torch = _torch()
    rng = np.random.default_rng(E * 100 + tokens + H)
    gu = random_blocks(rng, type_, E * 2 * I, H).reshape(-1)
    dn = random_blocks(rng, type_, E * H, I).reshape(-1)
    X = rng.normal(0, 1, (tokens, H)).astype(np.float32)
    wts = rng.uniform(0.1, 1, (tokens, k)).astype(np.float32)
    for routing in ("spread", "skewed"):
        ids = np.stack([rng.permutation(E)[:k] for _ in range(tokens)]).astype(np.int32)
        if routing == "skewed":
            ids[:, 0] = E - 1
            ids[ids[:, 1 % k] == E - 1, 1 % k] = 0 if k > 1 else E - 1
            ids[0, 0] = E  # out of range: contributes nothing
        say(f"few-pair experts type={type_} E={E} k={k} T={tokens} H={H} I={I} {routing}")
        valid = ids < E
        want = oracle.moe_routed(gu, dn, type_, E, H, I, X, np.where(valid, ids, 0).astype(np.int32),
                                 np.where(valid, wts, 0).astype(np.float32))
        bound = moe_bound(gu, dn, type_, E, H, I, X, ids, wts)
        got = []
        for offset in (0, 2):
            pools = []
            for w in (gu, dn):
                buf = torch.zeros(offset + w.size, dtype=torch.uint8, device="cuda:0")
                buf[offset:] = dev(w)
                pools.append(buf[offset:])
            Y = torch.full((tokens * H + 4,), 5.0, dtype=torch.float32, device="cuda:0")
            q3x.moe_routed(q3x.ExpertLinear(pools[0], E, 2 * I, H, type_), q3x.ExpertLinear(pools[1], E, H, I, type_),
                           dev(X), tokens, dev(ids), dev(wts), k, Y)
            y = host(Y)
            assert np.all(y[tokens * H:] == 5.0)
            got.append(y[:tokens * H].reshape(tokens, H))
        assert np.all(np.abs(got[0] - want) <= bound)
        # The two tile shapes: the same exact products in FP32 sums of another order.
        assert np.all(np.abs(got[0].astype(np.float64) - got[1]) <= 2 * bound)


@pytest.mark.parametrize("type_", [Q8_0, Q4_0])
@pytest.mark.parametrize("E,k,H,I,SI,tokens", [
    (64, 4, 256, 96, 96, 2), (64, 4, 256, 96, 64, 32), (64, 4, 256, 96, 96, 33),  # the per-token router's last count
    (40, 3, 128, 32, 32, 256), (40, 3, 128, 32, 32, 257),  # 1024 and 1028 pairs: one grouping workgroup and two
    (1023, 2, 64, 32, 32, 20), (1024, 2, 64, 64, 32, 20)])
def test_few_token_layer_routing(type_, E, k, H, I, SI, tokens):
    layers.test_moe_layer_parity(type_, E, H, I, SI, k, tokens)
