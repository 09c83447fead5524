"""The default choice on both sides of its lines.  (CPU: the choice alone, no kernel runs.)"""
import ctypes

import pytest

from host_arithmetic import load
from test_choice_per_device import Scratch

STRIP, BATCH = "s", "b"


@pytest.fixture(scope="module")
def chosen(tmp_path_factory):
    """(family, columns, tokens, K splits of a batch kernel) of the default choice on 256 CUs."""
    from lmdeploy_amd._lib import lib
    at = lib._ZN5w4a167algo_atEi
    at.restype, at.argtypes = ctypes.c_void_p, [ctypes.c_int]
    host = load(tmp_path_factory.mktemp("host"))
    host.describe.argtypes = [ctypes.c_void_p, ctypes.POINTER(ctypes.c_int)]

    def choice(N, K, T, nq=1):
        room, out = Scratch(None, 64 << 20, None, 1 << 16, 0, 256), (ctypes.c_int * 4)()
        host.describe(at(lib._ZN5w4a169algo_pickEiiiiRKNS_7ScratchEb(nq, N, T, K, ctypes.byref(room), 0)), out)
        return (chr(out[0]), *out[1:])

    return choice


@pytest.mark.parametrize("N,K,T,columns,splits", [
    (4096, 8192, 9, 16, 1), (4096, 10240, 16, 32, 2), (4096, 20352, 16, 32, 2), (4096, 20480, 16, 64, 4), (2048, 7040, 16, 16, 1),
    (2048, 7168, 9, 16, 2), (2048, 9216, 9, 32, 4), (1024, 4992, 16, 16, 1), (1024, 5120, 9, 16, 4), (1024, 8192, 8, 16, 4), (1536, 12288, 5, 32, 4), (5120, 10112, 12, 32, 1), (5120, 10240, 12, 48, 2), (8192, 16256, 16, 32, 1),
    (8192, 16384, 16, 64, 2), (12288, 28672, 16, 48, 1)])
def test_up_to_sixteen_tokens_split_deep_matrices(chosen, N, K, T, columns, splits):
    assert chosen(N, K, T) == (BATCH, columns, 16, splits)


@pytest.mark.parametrize("N,K,T,nq", [(1024, 8064, 8, 1), (1536, 12160, 8, 1), (4096, 28672, 8, 1), (2048, 4096, 5, 2), (512, 4096, 8, 4),
                                      (1024, 28672, 4, 1)])
def test_up_to_eight_tokens_stay_with_strips_below_the_line(chosen, N, K, T, nq):
    assert chosen(N, K, T, nq)[0] == STRIP


# (the second prices, asked alone, would move each of these to MFMA tiles, which round the weights)
@pytest.mark.parametrize("N,K,T", [(8064, 3328, 128), (12544, 3328, 81), (15104, 12544, 81), (17664, 13696, 128), (22144, 6784, 64),
                                   (22784, 7936, 100)])
def test_second_prices_move_nothing_to_rounded_weights(chosen, N, K, T):
    assert chosen(N, K, T)[0] == BATCH


@pytest.mark.parametrize("nq", [1, 2, 4])
def test_blocks_of_one_token_tile_end_where_they_are_priced(chosen, nq):
    assert chosen(4096, 4096, 24, nq) == (BATCH, 32, 16, 1)
    assert all(chosen(N, K, T, nq)[2] != 16 for N in (1024, 4096, 5120) for K in (1024, 4096, 11008) for T in (97, 100, 128, 129, 300)
               if chosen(N, K, T, nq)[0] == BATCH)


@pytest.mark.parametrize("N,K,T", [(3456, 4608, 351), (1728, 8320, 925), (9984, 2176, 118), (4480, 5120, 247)])
def test_tiles_of_64_by_64_are_not_taken_where_they_fill_the_chip_twice(chosen, N, K, T):
    assert chosen(N, K, T)[1:3] != (64, 64) or chosen(N, K, T)[0] == BATCH
