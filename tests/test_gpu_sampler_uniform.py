"""``rwkv7_sample_uniform`` (one set of parameters for every row) gives the tokens and
log-probabilities of ``rwkv7_sample`` with the same values in per-row arrays, bit for
bit: the same kernels, with the RNG counter equal to the row's index."""

import pytest
import torch

from rwkvtune_amd import _lib
from rwkvtune_amd import sampler as dsm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("temperature,top_p,top_k", [(1.0, 0.95, 0), (0.7, 0.85, 50), (0.0, 1.0, 0), (1e-6, 0.5, 1)])
@pytest.mark.parametrize("bias", [None, {3: 5.0, 70: -2.0}])
@pytest.mark.parametrize("rows,V", [(1, 65536), (33, 1000)])
def test_equals_per_row_arrays(gpu_device, dtype, temperature, top_p, top_k, bias, rows, V):
    print(f"[case] uniform sampling {dtype} t={temperature} p={top_p} k={top_k} bias={bias} {rows}x{V}", flush=True)
    g = torch.Generator(device=gpu_device).manual_seed(rows + V)
    x = (torch.randn(rows, V, generator=g, device=gpu_device) * 2).to(dtype)
    buf = dsm.SamplerBuffers(rows, gpu_device)
    buf.set_uniform(temperature, top_p, top_k)
    buf.set_bias(bias, rows)
    buf.rng_key.fill_(1)
    buf.rng_ctr.copy_(torch.arange(rows, dtype=torch.int32, device=gpu_device))
    tok = torch.empty(rows, dtype=torch.int64, device=gpu_device)
    lp = torch.empty(rows, dtype=torch.float32, device=gpu_device)
    dsm.sample_rows(x, buf, rule=dsm.RULE_BATCH, max_valid_id=V - 7, seed=5, out_tok=tok, out_logp=lp)
    old = dsm.TokenSampler._max_valid_token_id
    try:
        dsm.TokenSampler._max_valid_token_id = V - 7
        dsm.TokenSampler.manual_seed(5)
        t2, l2 = dsm.TokenSampler.sample_batch(x, temperature, top_p, top_k, bias)
    finally:
        dsm.TokenSampler._max_valid_token_id = old
    torch.cuda.synchronize()
    assert torch.equal(tok, t2) and torch.equal(lp, l2)


def test_arguments(gpu_device):
    print("[case] uniform sampling, arguments", flush=True)
    x = torch.zeros(2, 100, device=gpu_device)
    with pytest.raises(RuntimeError):
        dsm.TokenSampler.sample_batch(x, top_k=1 << 40)
    with pytest.raises(ValueError):
        _lib.call("rwkv7_sample_uniform", 0, 2, 100, None, 100, 0, -1, 1.0, 1.0, 0, None, None, None, 0, 0, None, None,
                  None)
    tok, lp = dsm.TokenSampler.sample_batch(x[:0])
    assert tok.shape == (0,) and lp.shape == (0,)
