"""The row pass of the selective log-softmax at the lengths where its pipeline begins
and ends, against float64."""

import pytest
import torch

from rwkvtune_amd.grpo_utils import selective_log_softmax

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("V", [8, 2040, 2048, 8184, 8192, 10240, 16384, 24576, 65535, 65536])
def test_log_softmax_row_lengths(gpu_device, dtype, V):
    """The pipelined row pass at the edges of its sets of four groups per thread (8,192 logits) and its group
    tail; the largest value in the first, a middle and the last group.  float32 sums: 1e-6 of |logsumexp|."""
    print(f"[case] log-softmax {dtype} V={V}", flush=True)
    g = torch.Generator(device=gpu_device).manual_seed(V)
    x = torch.randn(6, V, generator=g, device=gpu_device) * 3
    for i, j in enumerate((0, V // 2, V - 1)):
        x[i, j] = 40.0
    x[3] = -float("inf")
    x[3, V - 2] = 1.0
    x[4, 0], x[4, V - 1] = float("inf"), 1.0
    x[5] = x[5].abs() * -60.0
    x = x.to(dtype)
    idx = torch.tensor([0, 1, V - 1, V - 2, V - 1, V // 3], device=gpu_device)
    out = selective_log_softmax(x, idx)
    x64 = x.double()
    lse = torch.logsumexp(x64, -1)
    ref = x64.gather(1, idx[:, None])[:, 0] - lse
    tol = 1e-6 if dtype == torch.float32 else torch.finfo(dtype).eps
    for i in (0, 1, 2, 3, 5):
        # the result's own rounding, and (16 bits) the rounded logsumexp
        assert abs(float(out[i]) - float(ref[i])) <= tol * (abs(float(lse[i])) + abs(float(ref[i]))) + 1e-6, (i, out, ref)
    assert float(out[4]) == -float("inf")
