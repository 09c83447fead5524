"""The batch and tile kernels where they can go wrong: a last strip or tile that overlaps its neighbour, token counts
on both sides of every block and tile, one quantisation group (most waves of a batch workgroup have none), odd numbers of
groups (padding), K split unevenly, every group size, and outputs that are only four bytes aligned."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# against fp32 on the fp16 weights: the rounding of the result (2^-11 of it), of a weight that a decode kernel leaves
# unrounded (2^-11 of each product), and of fp32 sums of up to 1152 terms (below 2^-13 of the sum of products)
HALF_ULP = 2.0 ** -11


@pytest.fixture(scope="module")
def tm():
    import lmdeploy_amd.turbomind as tm
    return tm


def problem(tm, K, N, T, gs, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    words = lambda *size: torch.randint(-2 ** 31, 2 ** 31, size, dtype=torch.int32, device="cuda", generator=gen)
    s = (torch.randn((K // gs, N), device="cuda", generator=gen).abs() * 0.01 + 1e-3).half()
    qw = words(K, N // 8)
    A, Q = torch.empty_like(qw), torch.empty_like(s, dtype=torch.int32)
    tm.convert_s4_k_m8(A, Q, s, qw, s, words(K // gs, N // 8), N, K, gs)
    W = tm.dequantize_repacked(A, Q, N, K, gs).float()
    X = torch.randn((T, K), device="cuda", generator=gen).half()
    want = X.float() @ W
    allowed = HALF_ULP * want.abs() + (HALF_ULP + HALF_ULP / 4) * (X.float().abs() @ W.abs())
    return A, Q, X, want, allowed


@pytest.mark.parametrize("K,N", [(128, 272), (1152, 816)])
@pytest.mark.parametrize("T", [1, 15, 17, 33, 63, 65, 81, 97, 161, 225, 257])
def test_every_configuration_at_the_edges(tm, K, N, T):
    gemm = tm.GemmS4F16()
    A, Q, X, want, allowed = problem(tm, K, N, T, 128, 100 * T + N)
    ran = 0
    for algo in range(gemm.algo_count()):
        C = torch.full((T, N), float("nan"), dtype=torch.float16, device="cuda")
        try:
            gemm.Run(C, A, X, Q, N, T, K, 128, 0, algo)
        except tm.W4A16Error as e:
            assert e.code == -2, e
            continue
        assert ((C.float() - want).abs() <= allowed).all(), (K, N, T, algo)
        ran += 1
    assert ran >= 40


@pytest.mark.parametrize("gs", [64, 32])
@pytest.mark.parametrize("K,N", [(128, 272), (1152, 816), (640, 4096)])
def test_group_sizes_64_and_32_on_both_sides_of_every_hand_over(tm, gs, K, N):
    gemm = tm.GemmS4F16()
    for T in (16, 17, 31, 48, 65, 97, 129, 200, 257, 520):
        A, Q, X, want, allowed = problem(tm, K, N, T, gs, gs + T)
        C = torch.full((T, N), float("nan"), dtype=torch.float16, device="cuda")
        gemm.Run(C, A, X, Q, N, T, K, gs)
        assert ((C.float() - want).abs() <= allowed).all(), (gs, K, N, T)
        E = torch.full_like(C, float("nan"))
        tm.gemm_static(E, A, X, Q, N, T, K, gs)     # (may split K by another number: its own choice, the same bound)
        assert ((E.float() - want).abs() <= allowed).all(), (gs, K, N, T, "static")


@pytest.mark.parametrize("gs", [64, 32])
@pytest.mark.parametrize("T,N", [(9, 272), (17, 272), (33, 1088), (48, 4096), (48, 16384), (65, 4096), (100, 4096), (300, 4096)])
def test_subnormal_scales_of_small_groups(tm, gs, T, N):
    """A subnormal scale reads as zero whichever of a weight tile's groups it belongs to, in blocks of every width."""
    K   = 640
    gen = torch.Generator(device="cuda").manual_seed(T + N + gs)
    words = lambda *size: torch.randint(-2 ** 31, 2 ** 31, size, dtype=torch.int32, device="cuda", generator=gen)
    s = (torch.randn((K // gs, N), device="cuda", generator=gen).abs() * 0.01 + 1e-3).half()
    for col in range(7):  # another group in every seventh column, and the smallest normal scale beside them
        s[col % (128 // gs)::128 // gs, col::7] = 2.0 ** -15 if col < 6 else 2.0 ** -14
    qw = words(K, N // 8)
    A, Q = torch.empty_like(qw), torch.empty_like(s, dtype=torch.int32)
    tm.convert_s4_k_m8(A, Q, s, qw, s, words(K // gs, N // 8), N, K, gs)
    W = tm.dequantize_repacked(A, Q, N, K, gs).float()
    assert (W.view(K // gs, gs, N)[0, :, 0] == 0).all()
    X = (1000 * torch.randn((T, K), device="cuda", generator=gen)).half()  # (a product that is not left out would show)
    want = X.float() @ W
    allowed = HALF_ULP * want.abs() + (HALF_ULP + HALF_ULP / 4) * (X.float().abs() @ W.abs())
    C = torch.full((T, N), float("nan"), dtype=torch.float16, device="cuda")
    tm.GemmS4F16().Run(C, A, X, Q, N, T, K, gs)
    assert ((C.float() - want).abs() <= allowed).all()


@pytest.mark.parametrize("gs", [64, 32])
@pytest.mark.parametrize("K,N", [(4096 + 128, 272)] + [(384, 4096 * w - 896) for w in range(2, 9)] + [(128, 4096 * 9)])
def test_strips_of_every_width_with_small_groups(tm, gs, K, N):
    """One tile with sixteen waves, strips of two to eight tiles next to narrower ones, and several strips in turn."""
    gemm = tm.GemmS4F16()
    for T in (1, 4, 5, 8, 9, 16):
        A, Q, X, want, allowed = problem(tm, K, N, T, gs, gs + T + N)
        C = torch.full((T, N), float("nan"), dtype=torch.float16, device="cuda")
        gemm.Run(C, A, X, Q, N, T, K, gs)
        assert ((C.float() - want).abs() <= allowed).all(), (gs, K, N, T)


@pytest.mark.parametrize("T,N", [(6, 816), (12, 816), (20, 816), (32, 816), (33, 1024), (80, 768), (160, 128), (40, 64),
                                 (300, 48), (700, 816), (300, 192)])
def test_four_bytes_of_alignment(tm, T, N):
    """Up to 160 tokens, and beyond where the features are no multiple of 128."""
    K = 1152
    A, Q, X, want, allowed = problem(tm, K, N, T, 128, T)
    buf = torch.zeros(T * N + 8, dtype=torch.float16, device="cuda")
    C = buf[2:2 + T * N].view(T, N)
    tm.GemmS4F16().Run(C, A, X, Q, N, T, K, 128)
    assert ((C.float() - want).abs() <= allowed).all()
    assert (buf[:2] == 0).all() and (buf[2 + T * N:] == 0).all()


def test_column_blocks_of_the_batch_kernel_report_their_split(tm):
    """Eight waves of one, two or four workgroups share out K: three configurations, told apart by their slices."""
    gemm, T, N, K = tm.GemmS4F16(), 16, 1024, 4096
    A, Q, X, want, allowed = problem(tm, K, N, T, 128, 1)
    ms = gemm.Measure(torch.empty((T, N), dtype=torch.float16, device="cuda"), A, X, Q, N, T, K, 128)
    tiles = max(m.id for m in ms if m.kind == 1)
    blocks = [m for m in ms if m.kind == 0 and m.id > tiles]
    assert sorted((m.tile_n, m.slices) for m in blocks) == [(n, z) for n in (16, 32, 48, 64) for z in (8, 16, 32)]
    assert all(m.grid == -(-N // m.tile_n) * m.slices // 8 for m in blocks if m.feasible)
