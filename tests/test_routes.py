"""Which path a call takes: the rules of the dispatch as plain functions of addresses and sizes (no GPU, nothing is launched)."""
import ctypes as C

import pytest

from ferrotensor_amd import _lib


@pytest.fixture(scope="module")
def lib():
    return C.CDLL(_lib.LIB_PATH)


F32, F16 = 0, 1
MIB = 1 << 20


def group(*linears):
    """Descriptors at made-up addresses; each linear a dict of w, y, N and, if it has them, t, b, r, residual, rope_table."""
    descs = (_lib.LoraLinearDescC * len(linears))()
    for d, l in zip(descs, linears):
        d.w, d.w_dtype, d.y, d.N = l["w"], l.get("dtype", F32), l["y"], l["N"]
        d.t, d.b, d.residual, d.r = l.get("t"), l.get("b"), l.get("residual"), l.get("r", 0)
        d.rope_table, d.rope_seq = l.get("rope_table"), l.get("rope_seq", 0)
    return descs


@pytest.mark.parametrize("change,together", [
    ({}, True),
    ({"residual": 20 * MIB}, True),                        # its own output in place of its residual
    ({"t": 10 * MIB, "b": 40 * MIB, "r": 8}, False),       # the first linear's output as the rank-r factor
    ({"t": 10 * MIB - 4 * 64 * 8, "b": 40 * MIB, "r": 8}, True),   # ends where that output begins
    ({"t": 10 * MIB - 4 * 64 * 8 + 4, "b": 40 * MIB, "r": 8}, False),
    ({"residual": 10 * MIB}, False),                       # the first linear's output as residual
    ({"residual": 10 * MIB + 4 * (64 * 8 - 1)}, False),    # its last element
    ({"residual": 10 * MIB + 4 * 64 * 8}, True),
    ({"y": 10 * MIB}, False),                              # the same output twice
    ({"w": 10 * MIB}, False),
    ({"rope_table": 10 * MIB, "rope_seq": 4}, False),
    ({"t": 10 * MIB, "b": 40 * MIB, "r": 0}, True),        # a factor that is not used
])
@pytest.mark.parametrize("dtype", [F32, F16])
def test_linears_that_feed_each_other_do_not_share_a_launch(lib, change, together, dtype):
    first = {"w": 1 * MIB, "y": 10 * MIB, "N": 8, "dtype": dtype}
    second = dict({"w": 2 * MIB, "y": 20 * MIB, "N": 64, "dtype": dtype}, **change)
    M, K = C.c_size_t(64), C.c_size_t(96)
    for order in ((first, second), (second, first)):
        assert lib.ft_internal_group_apart(group(*order), C.c_size_t(2), M, K) == together, order
    assert lib.ft_internal_group_apart(group(second), C.c_size_t(1), M, K) == 1
