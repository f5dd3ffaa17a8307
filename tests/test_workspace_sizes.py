"""Workspace sizes on the host: a workspace sized once for a caller's most
tokens serves every smaller count of the same matrix or layer."""
import ctypes

import pytest

import qwen3x_amd as q3x
from tests.helpers import Q4_0, Q8_0


def _split_bytes(rows, cols, count):
    """Bytes of the partial sums that the call itself writes (q3x::gemm_split_bytes)."""
    f = q3x.lib()["_ZN3q3x16gemm_split_bytesEiii"]
    f.restype, f.argtypes = ctypes.c_size_t, [ctypes.c_int] * 3
    return f(rows, cols, count)


@pytest.mark.parametrize("rows,cols", [(12288, 4096), (4096, 12288), (5120, 17408), (1024, 5120), (6144, 2048),
                                       (24576, 5120), (700, 3072), (8300, 4128), (40000, 1024)])
def test_gemm_workspace_holds_smaller_counts(rows, cols):
    size = q3x.lib().q3x_hip_gemm_workspace_bytes
    most = [0]
    for count in range(1, 1301):
        most.append(max(most[-1], _split_bytes(rows, cols, count)))
    for count in list(range(2, 200, 3)) + [192, 193, 255, 256, 257, 511, 512, 640, 1300]:
        nbytes = size(Q8_0, rows, cols, count)
        assert nbytes == size(Q4_0, rows, cols, count)
        if count <= 192 or _split_bytes(rows, cols, count):
            assert nbytes >= most[count], count
        else:
            assert nbytes == 0, count


@pytest.mark.parametrize("E,k,H,I", [(256, 1, 32, 32), (512, 2, 64, 64), (512, 1, 256, 128), (1024, 8, 64, 32),
                                     (1024, 2, 128, 64), (8, 2, 1024, 512), (256, 8, 2048, 512)])
def test_moe_workspace_grows_with_the_tokens(E, k, H, I):
    """The few-pair tiles' table is longer than a larger call's 80-pair one;
    at 32 MiB the static scratch's limit decides between the two."""
    previous = 0
    for tokens in range(1, min(14 * E // k + 200, 6000)):
        nbytes = q3x.moe_workspace_bytes(tokens, E, k, H, I)
        assert nbytes >= previous, tokens
        previous = nbytes


@pytest.mark.parametrize("E,k,H,I,SI", [(8, 2, 1024, 512, 512), (8, 2, 1024, 512, 256), (1000, 1, 512, 1728, 1728),
                                        (64, 8, 1024, 96, 64)])
def test_moe_layer_workspace_grows_with_the_tokens(E, k, H, I, SI):
    weights = q3x.MoeLayerWeights(type=Q4_0, experts=E, top_k=k, H=H, I=I, shared_I=SI)
    previous = 0
    for tokens in range(1, 700):
        nbytes = q3x.lib().q3x_hip_moe_layer_workspace_bytes(ctypes.byref(weights), tokens)
        assert nbytes >= previous, tokens
        previous = nbytes
