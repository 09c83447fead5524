"""Where a workgroup of the batch and tile kernels finds its tile: the divisions by numbers of tiles and strips are products with
reciprocals, and the K splits shifts.  Every configuration on numbers of tiles that are prime, odd and multiples of four."""
import pytest
import torch


@pytest.mark.parametrize("bound_bits", [8, 16, 24, 31])
def test_reciprocals_are_exact_below_their_bound(bound_bits):
    """floor(2^32 / d) + 1, as the host makes them, wherever n d stays below 2^32 (elsewhere the kernels divide)."""
    import random
    rng = random.Random(bound_bits)
    for _ in range(20000):
        d = rng.randint(2, 1 << rng.randint(1, bound_bits))
        bound = (2 ** 32 - 1) // d
        by = 2 ** 32 // d + 1
        for n in (0, d - 1, d, bound, bound // d * d, bound // d * d - 1, rng.randint(0, bound)):
            if 0 <= n <= bound:
                assert n * by >> 32 == n // d, (n, d)


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
