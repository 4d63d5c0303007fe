"""The vector-ALU kernel for small outputs (32 x 32 blocks, k shared out between the waves of a workgroup): every number
of waves, block edges, chunk remainders, layouts, the masked / zero-sign / bit forms, partial tiles and batches."""
import numpy as np
import pytest

from helpers import assert_same_bits, to_device, to_host

pytestmark = pytest.mark.gpu

NPD = {"f32": np.float32, "f64": np.float64, "i32": np.int32, "u32": np.uint32}
PAIRS = [("minimum", "plus", "f32"), ("maximum", "minimum", "f64"), ("minimum", "multiplies", "f32"), ("maximum", "multiplies", "f64"),
         ("logical_or", "logical_and", "f64"), ("logical_or", "logical_and", "f32"), ("bit_xor", "bit_and", "u32"), ("minimum", "plus", "i32")]
# (m, n, k): four waves (few chunks), eight, sixteen; narrower than a block, whole blocks, one row and column more;
# k of one, of one chunk (16 floats, 8 doubles) and its neighbours, and of a chunk more than the waves share evenly
SHAPES = [(1, 1, 1), (31, 40, 7), (32, 32, 16), (33, 65, 17), (100, 37, 8), (64, 96, 129), (95, 33, 257), (160, 64, 1030), (33, 31, 2049)]


def _case(inputs, dtype, m, n, k, order, seed):
    npd = NPD[dtype]
    if dtype == "u32":
        return [inputs.words32(seed + (i << 40), r, c, o) for i, (r, c, o) in enumerate(zip((m, k, m), (k, n, n), order))]
    lo = 0 if dtype == "i32" else -3   # products of both signs and zeros of both signs
    return [inputs.integers(seed + (i << 40), r, c, lo, 8, npd, o) for i, (r, c, o) in enumerate(zip((m, k, m), (k, n, n), order))]


@pytest.mark.parametrize("pair", PAIRS)
@pytest.mark.parametrize("shape", SHAPES)
def test_small_outputs(oracle, lib, pair, shape):
    import torch
    import cuasr_amd
    from cuasr_amd import inputs
    add, mult, dt = pair
    ident, one = cuasr_amd.op_identity(add, dt, True), cuasr_amd.op_identity(mult, dt, True)
    for i, order in enumerate(("FFF", "CCC", "CFC", "FCF")):
        A, B, C = _case(inputs, dt, *shape, order, 31 + i)
        # (the host form always reads C: beta = the add's identity leaves it out only where identity (x) C is the identity
        # for every C -- not on int32, where it overflows, and not for products with numbers of either sign)
        for beta in (one,) if dt == "i32" or mult == "multiplies" else (one, ident):
            want = oracle.srgemm(add, mult, A, B, C, one, beta, ident)
            dD = to_device(np.zeros_like(C))
            cuasr_amd.srgemm(add, mult, to_device(A), to_device(B), to_device(C), dD, one, beta, ident, one, dtype=dt, kernel="valu")
            torch.cuda.synchronize()
            assert_same_bits(to_host(dD, dt), want, f"{pair} {shape} {order} beta={beta}")


@pytest.mark.parametrize("pair", PAIRS)
def test_small_outputs_in_place_in_slices_and_in_batches(oracle, lib, pair):
    import torch
    import cuasr_amd
    from cuasr_amd import inputs
    add, mult, dt = pair
    ident, one = cuasr_amd.op_identity(add, dt, True), cuasr_amd.op_identity(mult, dt, True)
    m, n, k = 70, 41, 530
    A, B, C = _case(inputs, dt, m, n, k, "CFC", 77)
    want = oracle.srgemm(add, mult, A, B, C, one, one, ident)
    dC = to_device(C)
    cuasr_amd.srgemm(add, mult, to_device(A), to_device(B), dC, dC, one, one, ident, one, dtype=dt, kernel="valu")   # D is C
    torch.cuda.synchronize()
    assert_same_bits(to_host(dC, dt), want, f"{pair} in place")
    for slices in (3, 4):   # (530 k in 4 slices of 144: the last one ragged)
        want = oracle.srgemm_splitk(add, mult, A, B, C, one, one, ident, one, slices)
        work = torch.empty(cuasr_amd.splitk_workspace_bytes(m, n, slices, dt) // 4, dtype=torch.int32, device="cuda")
        dD = to_device(np.zeros_like(C))
        cuasr_amd.srgemm_splitk(add, mult, to_device(A), to_device(B), to_device(C), dD, slices, work, one, one, ident, one, dtype=dt,
                                kernel="valu")
        torch.cuda.synchronize()
        got = to_host(dD, dt)
        if mult == "multiplies":   # the slices' zeros are folded at this library's slice boundaries: their sign is open
            assert np.array_equal(got, want)
        else:
            assert_same_bits(got, want, f"{pair} {slices} slices")
    for b, bm, bn, bk in ((37, 33, 20, 40), (300, 32, 32, 5)):
        ops = [_case(inputs, dt, bm, bn, bk, "CCC", 1000 + 7 * i) for i in range(b)]
        up = lambda j: torch.stack([to_device(np.ascontiguousarray(o[j])) for o in ops])
        dA, dB, dC = up(0), up(1), up(2)
        dD = torch.zeros_like(dC)
        cuasr_amd.srgemm_batched(add, mult, dA, dB, dC, dD, one, one, ident, one, dtype=dt, kernel="valu")
        torch.cuda.synchronize()
        for i in range(0, b, 9):
            want = oracle.srgemm(add, mult, *ops[i], one, one, ident)
            assert_same_bits(to_host(dD[i], dt), want, f"{pair} product {i} of {b}")


@pytest.mark.parametrize("pair", PAIRS)
@pytest.mark.parametrize("shape", [(1, 200, 300), (20, 97, 100), (500, 31, 70), (33, 2, 48), (17, 16, 129)])
def test_outputs_narrower_than_a_block(oracle, lib, pair, shape):
    """Vectors along k from clamped rows where an operand's rows are fewer than a block's, whole blocks on the other side;
    rows spaced wider than they are long."""
    import torch
    import cuasr_amd
    from cuasr_amd import inputs
    add, mult, dt = pair
    ident, one = cuasr_amd.op_identity(add, dt, True), cuasr_amd.op_identity(mult, dt, True)
    for i, order in enumerate(("FFF", "CCC", "CFC", "FCF")):
        A, B, C = _case(inputs, dt, *shape, order, 131 + i)
        want = oracle.srgemm(add, mult, A, B, C, one, one, ident)
        wide = []
        for x in (A, B):   # the leading dimension three elements more than it has to be
            t = to_device(x)
            base = t if x.flags.c_contiguous else t.t()
            room = torch.zeros(base.shape[0], base.shape[1] + 3, dtype=base.dtype, device="cuda")
            room[:, :base.shape[1]] = base
            wide.append(room[:, :base.shape[1]] if x.flags.c_contiguous else room[:, :base.shape[1]].t())
        dD = to_device(np.zeros_like(C))
        cuasr_amd.srgemm(add, mult, *wide, to_device(C), dD, one, one, ident, one, dtype=dt, kernel="valu")
        torch.cuda.synchronize()
        assert_same_bits(to_host(dD, dt), want, f"{pair} {shape} {order}")
