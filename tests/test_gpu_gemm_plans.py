"""GPU tests of every tile the GEMM plans run on past 32 tokens -- whole, split
over K, and with only the last round's tiles split -- each at sizes for which
the plan (q3x::gemm_plan) takes it, and of the paired gate and up launch on them
and on the few-token kernel.  Against float64 within the GEMM tests' bound."""
import ctypes

import pytest

import qwen3x_amd as q3x
from tests.helpers import Q4_0, Q8_0
from tests.test_gpu_parity import TOL, _torch, say

pytestmark = pytest.mark.gpu

SHAPES = ["128x256", "64x128", "64x64", "128x192", "64x128 K halves", "48x128", "80x256", "96x256"]  # X3Shape
WHOLE, SPLIT, TAIL = "whole", "split", "tail"
# The one-per-CU shapes can split the last round alone.
CASES = [(s, k) for s in ("128x256", "64x128 K halves", "80x256", "96x256") for k in (WHOLE, SPLIT, TAIL)] + \
        [(s, k) for s in ("48x128", "64x128", "64x64") for k in (WHOLE, SPLIT)]
ANY_BYTES = 2 ** 64 - 1


def _symbol(name, restype, *argtypes):
    f = q3x.lib()[name]
    f.restype, f.argtypes = restype, argtypes
    return f


def _plan(rows, cols, count, paired, workspace):
    out = (ctypes.c_int * 5)()
    _symbol("_ZN3q3x9gemm_planEiiibmPi", None, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_bool,
            ctypes.c_size_t, ctypes.c_void_p)(rows, cols, count, paired, workspace, out)
    shape, _, _, split, whole = out
    return SHAPES[shape], TAIL if whole else SPLIT if split > 1 else WHOLE


def _sizes(case, paired):
    """The least work (rows, cols, count, with a workspace) that the plan runs
    so.  Odd rows (the gate and up launch takes whole 128-row groups), K in
    uneven block counts, counts past the tiles' edges."""
    rows = (2176, 4224, 6272, 8320, 12416, 16512, 24704, 33408) if paired else \
        (1058, 2114, 4162, 6210, 8290, 12418, 16514, 24706, 33410)
    found = [(r * c * n, r, c, n, ws) for r in rows for c in (1056, 2080, 4128, 8224)
             for n in (37, 48, 53, 77, 90, 128, 150, 190, 230) for ws in (ANY_BYTES, 0)
             if _plan(r, c, n, paired, ws) == case]
    assert found, f"no sizes found for {case}"
    return min(found)[1:]


def _matrix(torch, g, type_, rows, cols, offset=0):
    """Blocks at `offset` bytes past an aligned start, and their float64 values."""
    n, block = rows * cols // 32, 34 if type_ == Q8_0 else 18
    b = torch.randint(0, 256, (n, block), dtype=torch.uint8, device="cuda:0", generator=g)
    d = torch.randn((n, 1), device="cuda:0", generator=g).mul_(0.02).to(torch.float16)
    b[:, :2] = d.view(torch.uint8)
    if type_ == Q8_0:
        v = b[:, 2:].contiguous().view(torch.int8).double()
    else:
        v = torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).double() - 8.0
    buf = torch.zeros(offset + n * block, dtype=torch.uint8, device="cuda:0")
    buf[offset:] = b.view(-1)
    return buf[offset:], (v * d.double()).view(rows, cols)


@pytest.mark.parametrize("type_", [Q8_0, Q4_0])
def test_dense_plans(type_):
    torch = _torch()
    g = torch.Generator(device="cuda:0")
    g.manual_seed(type_)
    for case in CASES + [("128x192", WHOLE)]:
        rows, cols, count, workspace = _sizes(case, False)
        say(f"dense {case[0]} {case[1]} type={type_} {rows}x{cols} count={count}")
        w, wd = _matrix(torch, g, type_, rows, cols)
        X = torch.randn((count, cols), device="cuda:0", generator=g)
        want = X.double() @ wd.T.contiguous()
        bound = TOL * X.double().norm(dim=1)[:, None] * wd.norm(dim=1)[None, :]
        lin = q3x.Linear(w, rows, cols, type_)
        nbytes = q3x.gemm_workspace_bytes(lin, count) if workspace else 0
        assert nbytes > 0 or case[1] == WHOLE
        ws = torch.full((nbytes + 64,), 0xA5, dtype=torch.uint8, device="cuda:0")
        Y = torch.full((count * rows + 8,), 3.0, device="cuda:0")
        again = torch.full_like(Y, 3.0)
        for out, add in ((Y, False), (again, False)):
            q3x.batch_mv_ws(lin, X, out, count, ws[:nbytes] if nbytes else None, add=add)
        got = Y[:count * rows].view(count, rows)
        assert bool((Y[count * rows:] == 3.0).all()) and bool((ws[nbytes:] == 0xA5).all())
        assert bool(((got.double() - want).abs() <= bound).all())
        assert torch.equal(Y.view(torch.int32), again.view(torch.int32))
        q3x.batch_mv_ws(lin, X, again, count, ws[:nbytes] if nbytes else None, add=True)  # exactly twice
        assert torch.equal(again[:count * rows].view(torch.int32), (got + got).view(-1).view(torch.int32))


def _gate_up(torch, g, type_, I, H, count, nbytes, offset=0):
    """q3x::gate_up_swiglu, the engine's dense feed-forward launch, on random
    operands: checks h = silu(gate x) * (up x) and returns its bits."""
    run = _symbol("_ZN3q3x14gate_up_swigluEPKvS1_jiiPKfiPfPvmP12ihipStream_t", ctypes.c_int, ctypes.c_void_p,
                  ctypes.c_void_p, ctypes.c_uint32, ctypes.c_int, ctypes.c_int, ctypes.c_void_p, ctypes.c_int,
                  ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_void_p)
    (gate, G), (up, U) = (_matrix(torch, g, type_, I, H, offset) for _ in range(2))
    X = torch.randn((count, H), device="cuda:0", generator=g)
    ws = torch.full((nbytes + 64,), 0xA5, dtype=torch.uint8, device="cuda:0")
    h = torch.full((count * I + 8,), 3.0, device="cuda:0")
    status = run(gate.data_ptr(), up.data_ptr(), type_, I, H, X.data_ptr(), count, h.data_ptr(),
                 ws.data_ptr() if nbytes else None, nbytes, torch.cuda.current_stream().cuda_stream)
    assert status == q3x.OK
    assert bool((h[count * I:] == 3.0).all()) and bool((ws[nbytes:] == 0xA5).all())
    Xd = X.double()
    a, b = Xd @ G.T.contiguous(), Xd @ U.T.contiguous()
    s = torch.sigmoid(a)
    xn = Xd.norm(dim=1)[:, None]
    # The products' errors to first order, and the activation's own rounding.
    bound = ((s * (1 + a * (1 - s)) * b).abs() * TOL * G.norm(dim=1)[None, :] * xn +
             (a * s).abs() * TOL * U.norm(dim=1)[None, :] * xn + 1e-6 * (a * s * b).abs() + 1e-37)
    got = h[:count * I].view(count, I)
    assert bool(((got.double() - a * s * b).abs() <= bound).all())
    return got


@pytest.mark.parametrize("type_", [Q8_0, Q4_0])
def test_paired_plans(type_):
    torch = _torch()
    g = torch.Generator(device="cuda:0")
    g.manual_seed(20 + type_)
    size = _symbol("_ZN3q3x30gate_up_swiglu_workspace_bytesEiii", ctypes.c_size_t, *[ctypes.c_int] * 3)
    for case in CASES:
        rows, cols, count, workspace = _sizes(case, True)
        nbytes = size(rows // 2, cols, count) if workspace else 0
        say(f"gate and up {case[0]} {case[1]} type={type_} {rows}x{cols} count={count} workspace={nbytes}")
        assert nbytes > 0 or case[1] == WHOLE
        _gate_up(torch, g, type_, rows // 2, cols, count, nbytes)
        if case[1] == SPLIT:  # half of it: the best plan that fits
            half = nbytes // 2 // 16 * 16
            say(f"  with {half} bytes: {_plan(rows, cols, count, True, half)}")
            _gate_up(torch, g, type_, rows // 2, cols, count, half)


@pytest.mark.parametrize("type_", [Q8_0, Q4_0])
def test_paired_few_tokens(type_):
    """2 to 32 tokens: whole and short K units, weights aligned to 16, 4 and 2
    bytes (the last on the general tiles)."""
    torch = _torch()
    g = torch.Generator(device="cuda:0")
    g.manual_seed(40 + type_)
    for I, H in ((192, 256), (4160, 1056), (64, 96), (1088, 2304)):
        for count in (2, 4, 5, 8, 9, 16, 17, 32, 33):
            for offset in (0, 4, 2):
                say(f"gate and up type={type_} {I}x{H} count={count} offset={offset}")
                _gate_up(torch, g, type_, I, H, count, 0, offset)
