"""Activations of just under 4 GiB, where 32-bit byte offsets into X end: the kernels that address X by 32-bit lane offsets
with a bias (the batch kernel, under its own ids and as the 32-token strips) on a matrix whose rows are short enough for the
bias to matter - 1864135 x 1152 halves are 256 bytes short of 4 GiB, and a row is shorter than the 3 KiB of the bias."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# 2^-11 of the result for its rounding and 2^-11 (plus a quarter for the fp32 sums) of the products for a rounded weight
HALF_ULP = 2.0 ** -11


@pytest.mark.parametrize("gs", [128, 64, 32])
def test_last_rows_of_four_gibibytes_of_activations(gs):
    import lmdeploy_amd.turbomind as tm
    T, K, N = 1864135, 1152, 16
    assert T * K * 2 < 2 ** 32 < (T - 1) * K * 2 + 3 * 1024 + 112
    gen = torch.Generator(device="cuda").manual_seed(gs)
    words = lambda *size: torch.randint(-2 ** 31, 2 ** 31, size, dtype=torch.int32, device="cuda", generator=gen)
    s = (torch.randn((K // gs, N), device="cuda", generator=gen).abs() * 0.01 + 1e-3).half()
    qw = words(K, N // 8)
    A, Q = torch.empty_like(qw), torch.empty_like(s, dtype=torch.int32)
    tm.convert_s4_k_m8(A, Q, s, qw, s, words(K // gs, N // 8), N, K, gs)
    W = tm.dequantize_repacked(A, Q, N, K, gs).float()
    X = torch.empty((T, K), dtype=torch.float16, device="cuda").normal_(generator=gen)
    gemm = tm.GemmS4F16()
    ids = [-1]
    if gs == 128:
        # (what an id is does not depend on the token count: asked at 32)
        few = gemm.Measure(torch.empty((32, N), dtype=torch.float16, device="cuda"), A, X, Q, N, 32, K, gs)
        gemm.clear_tuning()
        strips = [m.id for m in few if m.feasible and m.kind == 2 and m.tile_t == 32]
        assert strips
        ids += strips + [m.id for m in few if m.feasible and m.kind == 3 and m.slices == 1]
    for algo in ids:
        print("four GiB of activations: group size", gs, "kernel", algo, flush=True)
        C = torch.full((T, N), float("nan"), dtype=torch.float16, device="cuda")
        gemm.Run(C, A, X, Q, N, T, K, gs, 0, algo)
        for at in range(0, T, 1 << 17):
            x = X[at:at + (1 << 17)].float()
            want = x @ W
            allowed = HALF_ULP * want.abs() + (HALF_ULP + HALF_ULP / 4) * (x.abs() @ W.abs())
            assert ((C[at:at + (1 << 17)].float() - want).abs() <= allowed).all(), (gs, algo, at)
