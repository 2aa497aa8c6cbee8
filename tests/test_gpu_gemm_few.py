"""The grouped decode GEMM at 1 .. 8 rows (the kernel for a few rows ends at 7)
against float64: column counts off the 16-row tile, K tails and K shorter than a
tile, K ranges with the reduction launch, every epilogue, and the partial planes.

bf16 operands are exact and sums are float32: an element is its float64 value to a
bf16 ulp plus 64-bit-sum noise of K terms, 1e-6 * K^0.5 of the row's scale."""

import pytest
import torch

from rwkvtune_amd import _lib
from rwkvtune_amd.model import PackedWeight, RWKV7Model

pytestmark = pytest.mark.gpu


def epilogue(x, e):
    return torch.relu(x) ** 2 if e == 1 else torch.tanh(x) if e == 2 else torch.sigmoid(x) if e == 3 else x


@pytest.mark.parametrize("M", [1, 2, 5, 7, 8])
def test_few_rows(gpu_device, M):
    print(f"[case] grouped gemm, {M} rows", flush=True)
    g = torch.Generator(device=gpu_device).manual_seed(M)
    groups = [[(768, 768, 0), (96, 768, 2), (64, 768, 3), (3072, 768, 1)], [(768, 96, 0), (1, 8, 0), (17, 40, 1)],
              [(97, 4096, 0)], [(15, 72, 0), (300, 200, 2)], [(2048, 2048, 1)]]
    for grp in groups:
        probs, want = [], []
        for N, K, e in grp:
            # rows of a wider buffer whose other columns are not finite: nothing past K may be read into a sum
            wide = torch.full((M, K + 64), float("nan"), device=gpu_device, dtype=torch.bfloat16)
            A = wide[:, :K]
            A.copy_(torch.randn(M, K, generator=g, device=gpu_device))
            B = (torch.randn(N, K, generator=g, device=gpu_device) / K ** 0.5).bfloat16()
            C = torch.full((M, N + 3), 7.0, device=gpu_device, dtype=torch.bfloat16)
            probs.append((A, PackedWeight(B), C[:, :N], e))
            want.append((C, epilogue(A.double() @ B.double().t(), e), K))
        RWKV7Model._gemm_group(M, probs, _lib.stream_of(C))
        torch.cuda.synchronize()
        for (C, w, K), (N, _, _) in zip(want, grp):
            err = (C[:, :N].double() - w).abs()
            assert bool((err <= w.abs() * 2 ** -8 + 1e-6 * K ** 0.5).all()), (M, N, K, float(err.max()))
            assert bool((C[:, N:] == 7.0).all())


@pytest.mark.parametrize("M", [1, 3, 7])
@pytest.mark.parametrize("N,K", [(768, 768), (768, 3072), (2048, 8192), (50, 264), (16, 64)])
def test_few_rows_partials(gpu_device, M, N, K):
    print(f"[case] gemm partials, {M} rows {N} x {K}", flush=True)
    g = torch.Generator(device=gpu_device).manual_seed(N + K)
    A = torch.randn(M, K, generator=g, device=gpu_device).bfloat16()
    B = (torch.randn(N, K, generator=g, device=gpu_device) / K ** 0.5).bfloat16()
    ws, parts = RWKV7Model._gemm_partials(M, A, PackedWeight(B), _lib.stream_of(A))
    assert parts == _lib.load().rwkv7_gemm_decode_partial_count(M, N, K)
    torch.cuda.synchronize()
    got = ws[:parts * M * N].view(parts, M, N).double().sum(0)
    want = A.double() @ B.double().t()
    assert bool(((got - want).abs() <= 1e-6 * K ** 0.5).all())
