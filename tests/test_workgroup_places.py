"""Where a workgroup of the batch and tile kernels finds its tile: the divisions by numbers of tiles and strips are products with
reciprocals, and the K splits shifts.  Every configuration on numbers of tiles that are prime, odd and multiples of four."""
import ctypes
import random

import pytest
import torch

from host_arithmetic import load


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    lib = load(tmp_path_factory.mktemp("host"))
    lib.reciprocal_of.restype = lib.divide.restype = ctypes.c_uint
    lib.reciprocal_of.argtypes, lib.divide.argtypes = [ctypes.c_ulonglong, ctypes.c_uint], [ctypes.c_uint] * 3
    return lib


def check_divisions(lib, bound, d):
    """The launches' reciprocal of `d` for numbers below `bound`, at the places where a quotient changes."""
    by = lib.reciprocal_of(bound, d)
    at = {0, 1, d - 1, d, d + 1, bound - 1, bound // 2, bound // d * d, bound // d * d - 1, (bound // d - 1) * d - 1}
    for n in at:
        if 0 <= n < bound:
            assert lib.divide(n, d, by) == n // d, (n, d, bound, by)
    return by


@pytest.mark.parametrize("bits", [4, 8, 16, 24, 31])
def test_reciprocals_are_exact_below_their_bound(lib, bits):
    rng = random.Random(bits)
    for _ in range(5000):
        d = rng.randint(1, 1 << rng.randint(1, bits))
        check_divisions(lib, rng.randint(1, min(1 << 31, (2 ** 32 - 1) // d)), d)


@pytest.mark.parametrize("d", [1, 2, 3, 4, 7, 64, 97, 1 << 11, 65535, 65536, 65537, (1 << 20) - 1, 1 << 24])
def test_reciprocals_on_both_sides_of_their_bound(lib, d):
    most = 2 ** 32 // d         # bound x d below 2^32: a product; from there on: a division, which 1 stands for
    for bound in (most - 1, most, most + 1):
        if 1 <= bound < 2 ** 32:
            by = check_divisions(lib, bound, d)
            assert by == (0 if d == 1 else 2 ** 32 // d + 1 if bound * d < 2 ** 32 else 1)


@pytest.mark.parametrize("tiles_t,tiles_n", [(1, 1), (1, 172), (2, 7), (3, 97), (4, 1), (4, 86), (5, 64), (8, 33), (12, 5), (17, 13), (24, 40), (97, 101)])
def test_places_of_the_tile_kernels(lib, tiles_t, tiles_n):
    out = (ctypes.c_int * 5)()
    total = tiles_t * tiles_n
    for groups, splits in ((1, 1), (8, 1), (33, 1), (8, 2), (33, 2), (9, 4), (64, 4), (17, 8), (86, 8)):
        seen, ranges = set(), set()
        for split in range(splits):
            for i in range(total):
                id_ = (i & 7) * (total >> 3) + (i >> 3) if total % 8 == 0 else i        # (the kernels': runs for the XCDs)
                lib.tile_at(id_, tiles_t, tiles_n, groups, splits, split, out)
                t, n, z, begin, end = out
                assert 0 <= t < tiles_t and 0 <= n < tiles_n
                seen.add((t, n, z))
                ranges.add((z, begin, end))
        assert len(seen) == total * splits and len(ranges) == splits
        ends = [r[1:] for r in sorted(ranges)]
        assert ends[0][0] == 0 and ends[-1][1] == groups and all(a[1] == b[0] for a, b in zip(ends, ends[1:]))


@pytest.mark.parametrize("strips,tiles_t", [(1, 1), (1, 16), (7, 2), (16, 3), (97, 1), (86, 4), (33, 13), (128, 8), (251, 21)])
@pytest.mark.parametrize("splits", [1, 2, 4])
def test_places_of_the_batch_kernel(lib, strips, tiles_t, splits):
    out, seen = (ctypes.c_int * 3)(), set()
    for i in range(strips * tiles_t * splits):
        lib.batch_at(i, strips, tiles_t, splits, out)
        assert 0 <= out[0] < tiles_t and 0 <= out[1] < strips and 0 <= out[2] < splits
        seen.add(tuple(out))
    assert len(seen) == strips * tiles_t * splits


# (so many workgroups that a product with the reciprocal would not do: the kernels divide)
@pytest.mark.parametrize("strips,tiles_t,splits", [(3, 65537, 1), (1 << 12, 1 << 12, 4), (70001, 4099, 2), (1 << 11, 1 << 18, 1)])
def test_places_beyond_the_reciprocals(lib, strips, tiles_t, splits):
    rng, out, total = random.Random(strips), (ctypes.c_int * 3)(), strips * tiles_t * splits
    assert 1 in (lib.reciprocal_of(total, tiles_t), lib.reciprocal_of(strips * splits, strips)) and total < 2 ** 31
    for i in [0, 1, 7, 8, total - 1, total - 8] + [rng.randrange(total) for _ in range(20000)]:
        id_ = (i & 7) * (total >> 3) + (i >> 3) if total % 8 == 0 else i
        lib.batch_at(i, strips, tiles_t, splits, out)
        assert tuple(out) == (id_ % tiles_t, id_ // tiles_t % strips, id_ // tiles_t // strips)
        if splits == 1:
            lib.tile_at(id_, tiles_t, strips, 8, 1, 0, at := (ctypes.c_int * 5)())
            want = (id_ // 4 // strips * 4 + id_ % 4, id_ // 4 % strips) if tiles_t % 4 == 0 else (id_ % tiles_t, id_ // tiles_t)
            assert tuple(at)[:2] == want


@pytest.mark.gpu
@pytest.mark.parametrize("N,T", [(1040, 1000), (2288, 203), (528, 1343), (16 * 97, 17), (272, 2081)])
def test_every_tile_is_computed_once(N, T):
    import lmdeploy_amd.turbomind as tm
    K = 1024
    gen = torch.Generator(device="cuda").manual_seed(N + T)
    words = lambda *size: torch.randint(-2 ** 31, 2 ** 31, size, dtype=torch.int32, device="cuda", generator=gen)
    s = (torch.randn((K // 128, N), device="cuda", generator=gen).abs() * 0.01 + 1e-3).half()
    qw = words(K, N // 8)
    A, Q = torch.empty_like(qw), torch.empty_like(s, dtype=torch.int32)
    tm.convert_s4_k_m8(A, Q, s, qw, s, words(K // 128, N // 8), N, K, 128)
    X = torch.randn((T, K), device="cuda", generator=gen).half()
    want = X.double() @ tm.dequantize_repacked(A, Q, N, K).double()
    gemm, C = tm.GemmS4F16(), torch.empty((T, N), dtype=torch.float16, device="cuda")
    ms = gemm.Measure(C, A, X, Q, N, T, K, 128)
    gemm.clear_tuning()
    ids = [m.id for m in ms if m.feasible and m.kind in (0, 1, 3)]
    assert len(ids) > 60
    for algo in ids:
        C.fill_(float("nan"))
        gemm.Run(C, A, X, Q, N, T, K, 128, 0, algo)
        off = ((C.double() - want).abs() / want.std()).max().item()
        assert off < 2e-2, (algo, off)      # fp16 results up to five standard deviations (2^-9 there), and rounded weights
