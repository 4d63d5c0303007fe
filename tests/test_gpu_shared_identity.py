"""An additive identity that is not the add's own (the accumulation starts from whatever the descriptor names) where
several accumulators of one output meet: waves and groups of waves of a workgroup that share out k, workgroups that
share a slice of split-K, workgroups that share a tile.  In a sum or an exclusive or it counts once, not once each."""
import numpy as np
import pytest

from helpers import NP_OF, assert_same_bits, to_device, to_host

pytestmark = pytest.mark.gpu

IDENT, ONES = 0x5A5A1234, 0xFFFFFFFF


def _operands(m, n, k, dt, order="FCF"):
    from cuasr_amd import inputs
    ops = [inputs.words32(3 + (i << 40), r, c, o) for i, (r, c, o) in enumerate(zip((m, k, m), (k, n, n), order))]
    return [x.view(NP_OF[dt]) for x in ops]


def _signed(x, dt):
    return x - (1 << 32) if dt == "i32" and x >= 1 << 31 else x


# four, eight and sixteen waves on a 32 x 32 block; four and two groups of waves on a 64 x 64 tile, two on a 128 x 128 tile
SHAPES = [(33, 40, 7), (64, 60, 130), (96, 33, 1100), (860, 868, 300), (1300, 1340, 160), (2040, 2048, 128)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("add,mult,dt", [("bit_xor", "bit_and", "u32"), ("bit_xor", "bit_and", "i32"), ("plus", "multiplies", "i32"),
                                         ("bit_or", "bit_and", "u32"), ("minimum", "plus", "i32")])
def test_inside_a_workgroup(oracle, lib, add, mult, dt, shape):
    import torch
    import cuasr_amd
    m, n, k = shape
    A, B, C = _operands(m, n, k, dt)
    one = {"bit_and": _signed(ONES, dt), "multiplies": 1, "plus": 0}[mult]
    with np.errstate(over="ignore"):
        want = oracle.srgemm(add, mult, A, B, C, one, one, IDENT)
    dD = to_device(np.zeros_like(C))
    cuasr_amd.srgemm(add, mult, to_device(A), to_device(B), to_device(C), dD, one, one, IDENT, one, dtype=dt, kernel="valu")
    torch.cuda.synchronize()
    assert_same_bits(to_host(dD, dt), want, f"{add} {dt} {shape}")


@pytest.mark.parametrize("m,n,k,slices", [(64, 64, 8192, 2), (70, 41, 5000, 1)])
def test_workgroups_on_one_slice(oracle, lib, m, n, k, slices):
    import torch
    import cuasr_amd
    A, B, C = _operands(m, n, k, "u32")
    want = oracle.srgemm_splitk("bit_xor", "bit_and", A, B, C, ONES, ONES, IDENT, ONES, slices)
    work = torch.empty(cuasr_amd.splitk_workspace_bytes(m, n, slices, "u32") // 4, dtype=torch.int32, device="cuda")
    dD = to_device(np.zeros_like(C))
    cuasr_amd.srgemm_splitk("bit_xor", "bit_and", to_device(A), to_device(B), to_device(C), dD, slices, work, ONES, ONES, IDENT, ONES,
                            dtype="u32", kernel="valu")
    torch.cuda.synchronize()
    assert_same_bits(to_host(dD, "u32"), want, f"{slices} slices")


@pytest.mark.parametrize("source", [True, False])
def test_workgroups_on_one_tile(oracle, lib, source):
    """288 tiles of 256 x 128 for two workgroups per compute unit: most tiles are shared by several."""
    import torch
    import cuasr_amd
    m = n = 3072
    A, B, C = _operands(m, n, 64, "u32")
    beta = ONES if source else IDENT
    want = oracle.srgemm("bit_xor", "bit_and", A, B, C if source else np.zeros_like(C), ONES, beta, IDENT)
    dD = to_device(np.zeros_like(C))
    cuasr_amd.srgemm("bit_xor", "bit_and", to_device(A), to_device(B), to_device(C), dD, ONES, beta, IDENT, ONES, dtype="u32", kernel="streamk")
    torch.cuda.synchronize()
    assert_same_bits(to_host(dD, "u32"), want, f"source {source}")
