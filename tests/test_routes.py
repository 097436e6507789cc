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


AB, RANKED, RESIDUAL = (0, 0), (1, 0), (1, 1)


@pytest.mark.parametrize("half,terms,M,K,N,pays", [
    # where the f32 instruction was measured faster (256 CUs): short K
    (0, AB, 4096, 32, 576, 0), (1, AB, 4096, 32, 576, 0), (0, AB, 2048, 64, 576, 0), (1, AB, 2048, 64, 576, 0),
    (0, AB, 640, 64, 1536, 0), (0, AB, 1024, 128, 576, 0), (1, AB, 4096, 64, 1536, 0),
    (1, RANKED, 640, 128, 1536, 0), (1, RANKED, 1024, 64, 5120, 0), (1, RANKED, 2048, 128, 1536, 0),
    (1, RESIDUAL, 2048, 64, 5120, 0), (1, RESIDUAL, 4096, 128, 5120, 0), (1, RESIDUAL, 2048, 192, 1536, 0),
    # long K on few tiles
    (0, AB, 64, 4096, 256, 0), (0, AB, 128, 2560, 960, 0), (0, AB, 64, 16384, 2048, 0), (0, AB, 128, 16384, 2048, 0),
    # where the parts are: the same sizes with another b or more K or tiles, and the usual ones
    (1, AB, 640, 64, 1536, 1), (0, AB, 2048, 128, 576, 1), (1, AB, 1024, 128, 576, 1), (0, AB, 1024, 192, 576, 1),
    (1, AB, 8192, 64, 5120, 1), (0, AB, 8192, 64, 5120, 1), (1, RESIDUAL, 2048, 256, 1536, 1), (1, RANKED, 2048, 160, 1536, 1),
    (1, AB, 64, 16384, 2048, 1), (0, RANKED, 128, 2560, 960, 1), (0, AB, 192, 2560, 960, 1), (0, AB, 64, 2048, 2048, 1),
    (0, AB, 512, 16384, 2048, 1), (0, AB, 256, 2304, 512, 1), (1, RANKED, 2048, 960, 960, 1), (1, RESIDUAL, 2048, 576, 1536, 1),
    (0, AB, 1000, 960, 2560, 1), (0, AB, 17, 64, 64, 1), (1, AB, 17, 64, 64, 1),
])
def test_products_take_bf16_parts_where_those_are_faster(lib, half, terms, M, K, N, pays):
    assert lib.ft_internal_split_pays(C.c_size_t(256), half, *terms, C.c_size_t(M), C.c_size_t(K), C.c_size_t(N)) == pays


@pytest.mark.parametrize("gate_up,half,M,K,N,pays", [
    (0, 1, 1024, 64, 3072, 0), (0, 1, 1024, 128, 3072, 0), (0, 1, 2048, 64, 960, 0), (0, 1, 2048, 960, 1600, 1), (0, 1, 96, 64, 960, 1),
    (1, 1, 512, 32, 1536, 0), (1, 1, 512, 64, 5120, 0), (1, 1, 2048, 96, 5120, 0), (1, 0, 64, 8192, 1024, 0),
    (1, 1, 2048, 128, 5120, 1), (1, 1, 96, 960, 2560, 1), (1, 0, 256, 4096, 512, 1), (1, 0, 1024, 8192, 1024, 1),
])
def test_fused_launches_take_bf16_parts_where_those_are_faster(lib, gate_up, half, M, K, N, pays):
    assert lib.ft_internal_split_fused_pays(C.c_size_t(256), gate_up, half, C.c_size_t(M), C.c_size_t(K), C.c_size_t(N)) == pays


def on_parts(lib, B, Sq, Sk, H, Hkv, causal, forward_only=0):
    return lib.ft_internal_attention_split(*(C.c_size_t(x) for x in (256, B, Sq, Sk, H, Hkv)), causal, forward_only)


@pytest.mark.parametrize("B,S,H,Hkv,causal,pays", [
    # where the f32 kernels were measured faster, forward and backward together (256 CUs): large groups, short queries of
    # grouped heads, tiles half empty
    (4, 700, 32, 2, 1, 0), (4, 700, 32, 2, 0, 0), (3, 700, 32, 4, 1, 0), (8, 512, 32, 4, 1, 0), (3, 700, 32, 8, 1, 0),
    (24, 700, 8, 1, 0, 0), (16, 128, 32, 8, 1, 0), (8, 200, 32, 8, 1, 0), (24, 200, 9, 3, 0, 0), (24, 17, 32, 32, 1, 0),
    (24, 40, 32, 32, 1, 0), (24, 48, 32, 32, 1, 0), (13, 65, 32, 32, 0, 0), (12, 80, 32, 32, 1, 0), (1, 1024, 15, 5, 1, 0),
    (8, 256, 15, 5, 1, 0), (8, 256, 32, 8, 1, 0), (24, 300, 9, 3, 1, 0),
    # where the parts are
    (4, 1024, 15, 5, 1, 1), (8, 1024, 9, 3, 1, 1), (5, 1024, 15, 5, 1, 1), (8, 1024, 32, 32, 1, 1), (4, 384, 32, 8, 1, 1),
    (4, 700, 32, 8, 1, 1), (6, 384, 32, 8, 1, 1), (8, 1024, 32, 4, 1, 1), (8, 200, 32, 32, 1, 1),
    (8, 129, 32, 32, 1, 1), (12, 90, 32, 32, 1, 1), (24, 64, 32, 32, 1, 1), (16, 256, 15, 5, 0, 1), (12, 100, 32, 32, 1, 1),
    (3, 700, 32, 4, 0, 1), (8, 512, 32, 4, 0, 1),
])
def test_attention_backward_takes_bf16_parts_where_those_are_faster(lib, B, S, H, Hkv, causal, pays):
    assert on_parts(lib, B, S, S, H, Hkv, causal) == pays


@pytest.mark.parametrize("B,S,H,Hkv,pays", [(4, 8, 32, 32, 0), (1, 8, 9, 3, 1), (1, 23, 6, 2, 1), (1, 1024, 3, 1, 0), (1, 4096, 1, 1, 0), (1, 768, 9, 3, 0),
                                            (1, 40, 9, 3, 1), (1, 96, 15, 5, 1), (1, 384, 3, 1, 0), (1, 256, 3, 1, 1), (1, 1024, 15, 5, 1), (1, 2048, 15, 5, 1)])
def test_attention_forward_alone_takes_bf16_parts_where_those_are_faster(lib, B, S, H, Hkv, pays):
    assert on_parts(lib, B, S, S, H, Hkv, 1, 1) == pays
