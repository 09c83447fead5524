"""Where the default choice scales sums in fp32, results are those of unrounded weights: sizes whose kernels have always
done so must not be handed to an MFMA tile, which rounds (q - z) s to fp16.

Every row of X holds three ones inside one quantisation group, so the exact result is s (i1 + i2 + i3), an 11-bit number
times a 6-bit one: fp32 holds it, and a kernel that scales in fp32 returns its rounding to fp16, bit for bit.  A kernel that
rounds each weight first is off by an ulp in a good part of the outputs."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tm():
    import lmdeploy_amd.turbomind as tm
    return tm


def problem(tm, K, N, T, gs):
    gen = torch.Generator(device="cuda").manual_seed(K + N + T)
    words = lambda *size: torch.randint(-2 ** 31, 2 ** 31, size, dtype=torch.int32, device="cuda", generator=gen)
    s = (torch.randn((K // gs, N), device="cuda", generator=gen).abs() * 0.01 + 1e-3).half()
    qw, qz = words(K, N // 8), words(K // gs, N // 8)
    A, Q = torch.empty_like(qw), torch.empty_like(s, dtype=torch.int32)
    tm.convert_s4_k_m8(A, Q, s, qw, s, qz, N, K, gs)
    nibble = torch.tensor([0, 4, 1, 5, 2, 6, 3, 7], device="cuda") * 4          # of the eight columns of a word
    nibbles = lambda w: (w.unsqueeze(-1) >> nibble & 15).reshape(w.size(0), -1)
    group = torch.randint(K // gs, (T,), device="cuda", generator=gen)
    inside = torch.rand((T, gs), device="cuda", generator=gen).topk(3).indices    # three different rows of the group
    rows = group[:, None] * gs + inside
    X = torch.zeros((T, K), dtype=torch.float16, device="cuda").scatter_(1, rows, 1.0)
    whole = -3 * nibbles(qz)[group]
    for j in range(3):
        whole += nibbles(qw[rows[:, j]])
    want = (whole.double() * s[group].double()).half()
    rounded = sum(((nibbles(qw[rows[:, j]]) - nibbles(qz)[group]).double() * s[group].double()).half().double() for j in range(3)).half()
    return A, Q, X, want, rounded


def check(C, want, rounded, what):
    off = (C != want).sum().item()
    assert (rounded != want).float().mean().item() > 0.05        # (the inputs tell the two apart)
    assert off == 0, (what, off, want.numel())


# N an odd multiple of 64: streamed by strips and column blocks until 64 x 64 tiles were priced below them
@pytest.mark.parametrize("K,N,T", [(4096, 10944, 3329), (8192, 10176, 3329), (2048, 8256, 3329), (1664, 9920, 641), (1664, 9920, 1900),
                                   (4096, 18880, 7795), (11904, 11968, 4346), (2176, 576, 5901), (1664, 960, 2302), (1152, 128, 9592)])
def test_sizes_that_were_never_rounded(tm, K, N, T):
    A, Q, X, want, rounded = problem(tm, K, N, T, 128)
    C = torch.full((T, N), float("nan"), dtype=torch.float16, device="cuda")
    tm.GemmS4F16().Run(C, A, X, Q, N, T, K, 128)
    check(C, want, rounded, (K, N, T))
    # ... and whose outputs (and residuals) need four bytes of alignment, no more
    buf = torch.zeros(2 * T * N + 8, dtype=torch.float16, device="cuda")
    D, R = buf[2:2 + T * N].view(T, N), buf[2 + T * N:2 + 2 * T * N].view(T, N)
    for kind, res in ((0, None), (2, R)):
        D.fill_(float("nan"))
        tm.GemmS4F16().Run(D, A, X, Q, N, T, K, 128, kind, residual=res)
        check(D, want, rounded, (K, N, T, kind))


# the entry point without a handle has less room to split K, which made its tiles slower and its streaming range longer
@pytest.mark.parametrize("K,N,T", [(2176, 17792, 79), (2176, 10432, 4223), (1792, 17472, 1899)])
def test_sizes_that_were_never_rounded_without_a_handle(tm, K, N, T):
    A, Q, X, want, rounded = problem(tm, K, N, T, 128)
    C = torch.full((T, N), float("nan"), dtype=torch.float16, device="cuda")
    tm.gemm_static(C, A, X, Q, N, T, K, 128)
    check(C, want, rounded, (K, N, T))


# ... and so does a handle that has not split K yet while the stream is being captured: it cannot allocate its workspace then
@pytest.mark.parametrize("K,N,T", [(4736, 704, 3159), (8704, 448, 4763)])
def test_sizes_that_were_never_rounded_without_a_workspace(tm, K, N, T):
    A, Q, X, want, rounded = problem(tm, K, N, T, 128)
    C = torch.full((T, N), float("nan"), dtype=torch.float16, device="cuda")
    gemm, stream, g = tm.GemmS4F16(), torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=stream):
        gemm.Run(C, A, X, Q, N, T, K, 128, stream=torch.cuda.current_stream().cuda_stream)
    for _ in range(3):
        C.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        check(C, want, rounded, (K, N, T))


@pytest.mark.parametrize("gs", [64, 32])
@pytest.mark.parametrize("T", [33, 300, 1000])
def test_small_groups_with_outputs_of_four_bytes_of_alignment(tm, gs, T):
    """The rounding tile of group sizes 64 and 32 never took such outputs; SiLU pairs always fitted."""
    K, N = 4096, 4096
    A, Q, X, want, rounded = problem(tm, K, N, T, gs)
    buf = torch.zeros(2 * T * N + 8, dtype=torch.float16, device="cuda")
    low, high = buf[2:2 + T * N].view(T, N), buf[4 + T * N:4 + 2 * T * N].view(T, N)
    assert low.data_ptr() % 8 == 4 and high.data_ptr() % 8 == 0
    aligned = torch.zeros((T, N), dtype=torch.float16, device="cuda")
    for kind, C, R in ((0, low, None), (2, low, high), (2, aligned, low)):
        C.fill_(float("nan"))
        if R is not None:
            R.zero_()
        tm.GemmS4F16().Run(C, A, X, Q, N, T, K, gs, kind, residual=R)
        check(C, want, rounded, (gs, T, kind))
        if R is not None:
            R.zero_()
        C.fill_(float("nan"))
        tm.gemm_static(C, A, X, Q, N, T, K, gs, kind, residual=R)
        check(C, want, rounded, (gs, T, kind, "static"))
