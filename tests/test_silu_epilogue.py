"""The SiLU epilogue of the batch kernel and of all MFMA tiles divides: the same gate and up sums give the same halves."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gs", [128, 64, 32])
def test_silu_is_the_same_in_batch_and_tile_kernels(gs):
    """One activation of one per token: the sums are single weights, exact in fp16 whether a kernel rounds weights or not, and
    only the epilogue is left.  (A reciprocal that is an ulp of fp32 off moves about one half in ten thousand.)"""
    import lmdeploy_amd.turbomind as tm
    K, N, T = 4096, 8192, 600
    gen = torch.Generator(device="cuda").manual_seed(gs)
    words = lambda *size: torch.randint(-2 ** 31, 2 ** 31, size, dtype=torch.int32, device="cuda", generator=gen)
    s = (torch.randn((K // gs, N), device="cuda", generator=gen).abs() * 0.3 + 1e-2).half()
    qw = words(K, N // 8)
    A, Q = torch.empty_like(qw), torch.empty_like(s, dtype=torch.int32)
    tm.convert_s4_k_m8(A, Q, s, qw, s, words(K // gs, N // 8), N, K, gs)
    X = torch.zeros((T, K), dtype=torch.float16, device="cuda")
    X[torch.arange(T, device="cuda"), torch.randperm(K, device="cuda", generator=gen)[:T]] = 1.0
    gemm = tm.GemmS4F16()
    run = lambda x, algo: (out := torch.full((x.size(0), N // 2), float("nan"), dtype=torch.float16, device="cuda"),
                           gemm.Run(out, A, x, Q, N, x.size(0), K, gs, gemm.kFusedSiluFfn, algo))[0]
    few = torch.cat([run(X[i:i + 40], -1) for i in range(0, T, 40)])      # (of forty tokens: the batch kernel)
    assert torch.isfinite(few).all() and few.abs().mean() > 0.1
    ids = [-1]
    if gs == 128:
        ms = gemm.Measure(torch.empty((T, N), dtype=torch.float16, device="cuda"), A, X, Q, N, T, K, gs)
        gemm.clear_tuning()
        ids += [m.id for m in ms if m.feasible and m.kind in (1, 3) and m.slices == 1]
        assert len(ids) > 20
    for algo in ids:
        off = (run(X, algo) != few).sum().item()
        assert off == 0, (gs, algo, off, few.numel())


@pytest.mark.parametrize("gs", [128, 64, 32])
def test_silu_of_every_finite_half_and_of_infinities(gs):
    """Gates that run through all finite halves, up projections of one and of three, and infinite gates and up projections."""
    import lmdeploy_amd.turbomind as tm
    K, N = 256, 256
    q = torch.zeros((K, N), dtype=torch.int32, device="cuda")       # logical weights; zero point 0, scale 1
    q[0, 0::2] = 1                                                  # every gate is X[:, 0], every up projection X[:, 1]
    q[1, 1::2] = 1
    q[2, :] = 1                                                     # X[:, 2] is both
    order = torch.tensor([0, 2, 4, 6, 1, 3, 5, 7], device="cuda")
    words = (q.view(K, N // 8, 8)[:, :, order] << (4 * torch.arange(8, device="cuda"))).sum(-1).to(torch.int32)
    one = torch.ones((K // gs, N), dtype=torch.float16, device="cuda")
    A, Q = torch.empty_like(words), torch.empty_like(one, dtype=torch.int32)
    tm.convert_s4_k_m8(A, Q, one, words, one, torch.zeros((K // gs, N // 8), dtype=torch.int32, device="cuda"), N, K, gs)
    halves = torch.arange(-2 ** 15, 2 ** 15, dtype=torch.int32, device="cuda").to(torch.int16).view(torch.float16)
    halves = halves[halves.isfinite()]
    X = torch.zeros((2 * halves.numel() + 2, K), dtype=torch.float16, device="cuda")
    X[:-2, 0], X[:-2, 1] = halves.repeat(2), torch.tensor([1.0, 3.0], device="cuda").half().repeat_interleave(halves.numel())
    X[-2, 2], X[-1, 2] = float("inf"), float("-inf")
    gemm, T = tm.GemmS4F16(), X.size(0)
    few = torch.empty((T, N // 2), dtype=torch.float16, device="cuda")
    some = 4000 if gs == 128 else 30                                # (what the batch kernel is given, the last piece too)
    for i in range(0, T, some):
        gemm.Run(few[i:i + some], A, X[i:i + some], Q, N, min(some, T - i), K, gs, gemm.kFusedSiluFfn)
    assert (few[-2] == float("inf")).all() and few[-1].isnan().all()
    gate = halves.double().repeat(2)
    want = gate / (1 + torch.exp(-gate)) * X[:-2, 1].double()
    assert torch.allclose(few[:-2, 0].double(), want.clamp(-65504, 65504).where(want < 65520, float("inf")), rtol=2e-3, atol=6e-8)
    if gs == 128:
        ms = gemm.Measure(torch.empty((600, N // 2), dtype=torch.float16, device="cuda"), A, X, Q, N, 600, K, gs, gemm.kFusedSiluFfn)
        gemm.clear_tuning()
        ids = [m.id for m in ms if m.feasible and m.kind == 1 and m.slices == 1]
        assert len(ids) > 10
    else:
        ids = [-1]                                                  # this many tokens run on tiles
    for algo in ids:
        got = torch.empty_like(few)
        gemm.Run(got, A, X, Q, N, T, K, gs, gemm.kFusedSiluFfn, algo)
        off = ((got != few) & ~(got.isnan() & few.isnan())).sum().item()
        assert off == 0, (gs, algo, off)
