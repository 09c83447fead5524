"""The arrival counters of `w4a16_gemm_static` after a misuse: calls that overlapped against the rules, or a launch that was
abandoned, leave counts behind, and neither the next launch nor a graph's next replay may take them for its own.  What such
calls leave is written into the counters from the host, between launches; the launches themselves are ordinary ones."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

TAG_SHIFT = 12      # a tagged counter word: the launch's tag above, arrivals below (w4a16_internal.h, kEpochShift)


class Scratch(ctypes.Structure):
    """w4a16::Scratch."""
    _fields_ = [("ws", ctypes.c_void_p), ("ws_bytes", ctypes.c_size_t), ("cnt", ctypes.c_void_p), ("cnt_len", ctypes.c_int),
                ("epoch", ctypes.c_int), ("cus", ctypes.c_int)]


def scratch(lib):
    fn = getattr(lib, "_ZN5w4a1614static_scratchEPNS_7ScratchE")
    fn.restype, fn.argtypes = ctypes.c_int, [ctypes.POINTER(Scratch)]
    s = Scratch()
    assert fn(ctypes.byref(s)) == 0 and s.cnt and s.cnt_len == 4096
    return s


def write_counters(lib, words):
    """All three parts of the counters (w4a16_internal.h, kStaticCounters): eight bytes each of launches made at once, tagged words of
    four, and eight each of recorded launches."""
    s = scratch(lib)
    assert len(words) == 5 * s.cnt_len
    torch.cuda.synchronize()
    fn = lib.hipMemcpy
    fn.restype, fn.argtypes = ctypes.c_int, [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int]
    assert fn(s.cnt, (ctypes.c_int * len(words))(*words), 4 * len(words), 1) == 0      # host to device
    torch.cuda.synchronize()


def leave_behind(lib, word):
    """`word` >> TAG_SHIFT: the tag of a launch, and below it how many arrivals of it every counter holds."""
    n, count = scratch(lib).cnt_len, word & (1 << TAG_SHIFT) - 1
    write_counters(lib, [count, (word >> TAG_SHIFT) * count] * n + [word] * n + [word] * 2 * n)


# a batch kernel as column blocks, the same as blocks of some dozen tokens, column blocks, and MFMA tiles; all split K
@pytest.mark.parametrize("K,N,T,kind", [(8192, 1024, 16, None), (4224, 1024, 100, 3), (5632, 1024, 12, 0), (4224, 1024, 100, 1)])
def test_counts_left_behind_concern_no_later_launch_or_replay(K, N, T, kind):
    import lmdeploy_amd.turbomind as tm
    from lmdeploy_amd._lib import lib
    gen = torch.Generator(device="cuda").manual_seed(K + T)
    words = lambda *size: torch.randint(-2 ** 31, 2 ** 31, size, dtype=torch.int32, device="cuda", generator=gen)
    s = (torch.randn((K // 128, N), device="cuda", generator=gen).abs() * 0.01 + 1e-3).half()
    qw = words(K, N // 8)
    A, Q = torch.empty_like(qw), torch.empty_like(s, dtype=torch.int32)
    tm.convert_s4_k_m8(A, Q, s, qw, s, words(K // 128, N // 8), N, K, 128)
    X = torch.randn((T, K), device="cuda", generator=gen).half()
    gemm = tm.GemmS4F16()
    C = torch.empty((T, N), dtype=torch.float16, device="cuda")
    ids = [-1]
    if kind is not None:
        ms = gemm.Measure(C, A, X, Q, N, T, K, 128)
        gemm.clear_tuning()
        blocks = lambda m: -(-N // m.tile_n) * -(-T // m.tile_t)
        ids = [m.id for m in ms if m.feasible and m.kind == kind and m.grid > blocks(m)][:3]
        assert ids
    for algo in ids:
        stream = torch.cuda.Stream()
        g = torch.cuda.CUDAGraph()
        tm.gemm_static(C, A, X, Q, N, T, K, 128, 0, algo)
        with torch.cuda.graph(g, stream=stream):
            tm.gemm_static(C, A, X, Q, N, T, K, 128, 0, algo, stream=torch.cuda.current_stream().cuda_stream)
        captured = scratch(lib).epoch - 1
        E, H = torch.empty_like(C), torch.empty_like(C)
        for word in (0, 1, 5, *(captured << TAG_SHIFT | n for n in (1, 2, 3, 5, 1)), (captured + 7) << TAG_SHIFT | 1, 0):
            X.copy_(torch.randn((T, K), device="cuda", generator=gen).half())
            gemm.Run(H, A, X, Q, N, T, K, 128, 0, algo if algo >= 0 else gemm.pick(N, T, K))
            leave_behind(lib, word)
            C.fill_(float("nan"))
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(C.view(torch.int16), H.view(torch.int16)), ("replay", algo, word >> TAG_SHIFT, word & 4095)
            leave_behind(lib, word)
            tm.gemm_static(E, A, X, Q, N, T, K, 128, 0, algo)
            torch.cuda.synchronize()
            assert torch.equal(E.view(torch.int16), H.view(torch.int16)), ("call", algo, word >> TAG_SHIFT, word & 4095)


@pytest.mark.parametrize("splits_of", [(8192, 1024, 16), (4224, 1024, 100)])
def test_second_counters_left_behind(splits_of):
    """A count that did not start from zero is taken on a second set of counters: whatever those hold, and the call after it."""
    import lmdeploy_amd.turbomind as tm
    from lmdeploy_amd._lib import lib
    K, N, T = splits_of
    gen = torch.Generator(device="cuda").manual_seed(T)
    words = lambda *size: torch.randint(-2 ** 31, 2 ** 31, size, dtype=torch.int32, device="cuda", generator=gen)
    s = (torch.randn((K // 128, N), device="cuda", generator=gen).abs() * 0.01 + 1e-3).half()
    qw = words(K, N // 8)
    A, Q = torch.empty_like(qw), torch.empty_like(s, dtype=torch.int32)
    tm.convert_s4_k_m8(A, Q, s, qw, s, words(K // 128, N // 8), N, K, 128)
    X, H, E = torch.randn((T, K), device="cuda", generator=gen).half(), *torch.empty((2, T, N), dtype=torch.float16, device="cuda")
    gemm = tm.GemmS4F16()
    gemm.Run(H, A, X, Q, N, T, K, 128)
    for first, second in ((0, 3), (3, 0), (3, 3), (1 << 20, -1), (-1, 2 << TAG_SHIFT | 1)):
        n = scratch(lib).cnt_len
        write_counters(lib, [first, first] * n + [second] * n + [0] * 2 * n)
        for call in range(3):
            E.fill_(float("nan"))
            tm.gemm_static(E, A, X, Q, N, T, K, 128)
            torch.cuda.synchronize()
            assert torch.equal(E.view(torch.int16), H.view(torch.int16)), (first, second, call)
