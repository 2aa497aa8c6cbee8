"""The segmented walk of the chunked WKV7 forward (few (sequence, head) pairs:
state pass, scan, full pass) against the same call without a workspace (one block
per pair over the whole sequence) and the float64 recurrence.

Both sides take the same products in the same chunks; only the state at a
segment's start differs, by the composition of the segments' maps (hi / lo operand
parts, ~1e-5 of the state's scale).  y: one ulp of its type + 1e-4 of max|y|;
states, sa and checkpoints (float32): 1e-4 of their largest magnitude.
"""

import pytest
import torch

from oracle import wkv7 as ow
from rwkvtune_amd import _lib
from rwkvtune_amd import operators as ops
from rwkvtune_amd.workloads import cu_seqlens_of, wkv_inputs, wkv_state

pytestmark = pytest.mark.gpu


def close(a, b, frac, ulp=0.0):
    a, b = a.double().cpu(), b.double().cpu()
    return bool(((a - b).abs() <= ulp * b.abs() + frac * float(b.abs().max()) + 1e-12).all())


def unsplit_prefill(pool, slot, cu, ins, total):
    """rwkv7_wkv_prefill, which takes no workspace."""
    y = torch.empty_like(ins[0])
    _lib.call("rwkv7_wkv_prefill", _lib.dtype_code(y.dtype), cu.numel() - 1, pool.shape[1], total, _lib.ptr(cu),
              _lib.ptr(slot), _lib.ptr(pool), pool.shape[0], *(_lib.ptr(t) for t in ins), _lib.ptr(y), 0,
              _lib.stream_of(y))
    return y


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,lens", [(4, [129]), (4, [160, 1, 512, 31]), (12, [1000]), (20, [700, 64, 400]),
                                    (4, [0, 733, 32]), (40, [2048, 33])])
def test_ragged_prefill(gpu_device, dtype, H, lens):
    print(f"[case] segmented prefill {dtype} H={H} lens={lens}", flush=True)
    total, n = sum(lens), len(lens)
    assert ops._segment_ws(dtype, n, H, 0, total, 1, gpu_device)[1] > 0
    ins = [x.to(gpu_device) for x in wkv_inputs((total,), H, seed=total, dtype=dtype).as_tuple()]
    ins[1][total // 2, 5] = 1.0  # a chunk below the matrix form's log-decay floor
    cu = torch.tensor(cu_seqlens_of(lens), dtype=torch.int32, device=gpu_device)
    slot = torch.tensor([n - 1 - i for i in range(n)], dtype=torch.int32, device=gpu_device)
    pool0 = wkv_state(n + 1, H).to(gpu_device)
    pool = pool0.clone()
    y = ops.wkv7_prefill(pool, slot, cu, *ins)
    ref = pool0.clone()
    y_ref = unsplit_prefill(ref, slot, cu, ins, total)
    torch.cuda.synchronize()
    assert close(y, y_ref, 1e-4, torch.finfo(dtype).eps) and close(pool, ref, 1e-4)
    assert torch.equal(pool[n], pool0[n])  # a slot that no sequence uses
    # the longest sequence against the recurrence
    i = max(range(n), key=lambda j: lens[j])
    lo, hi = cu_seqlens_of(lens)[i], cu_seqlens_of(lens)[i + 1]
    one = [x[None, lo:hi].double().cpu() for x in ins]
    y64, s64 = ow.wkv7_rowwise(*one, state=pool0[slot[i].item()][None].double().cpu())
    assert close(y[lo:hi], y64[0], 1e-3, torch.finfo(dtype).eps) and close(pool[slot[i].item()], s64[0], 1e-4)


def test_offsets_that_decrease(gpu_device):
    """A range that ends before it starts is skipped, also where the others then cover more rows than
    there are (more segments than blocks): as without a workspace."""
    H, total = 4, 2560
    ins = [x.to(gpu_device) for x in wkv_inputs((total,), H, seed=5).as_tuple()]
    cu = torch.tensor([0, 2400, 160, 2560, 40, 2520], dtype=torch.int32, device=gpu_device)
    pool0 = wkv_state(5, H).to(gpu_device)
    pool, ref = pool0.clone(), pool0.clone()
    print("[case] segmented prefill, decreasing offsets", flush=True)
    ops.wkv7_prefill(pool, None, cu, *ins)
    unsplit_prefill(ref, None, cu, ins, total)
    torch.cuda.synchronize()
    assert close(pool, ref, 1e-4) and torch.equal(pool[1], pool0[1])


@pytest.mark.parametrize("B,T,H", [(1, 513, 4), (2, 200, 12), (4, 1024, 32), (5, 1100, 32)])
@pytest.mark.parametrize("alias", [False, True])
def test_training_forward(gpu_device, B, T, H, alias):
    """y, sa, checkpoints and the final state; the final state may be written over the initial one."""
    print(f"[case] segmented training forward B={B} T={T} H={H} alias={alias}", flush=True)
    dtype = torch.bfloat16
    assert ops._segment_ws(dtype, B, H, T, B * T, 2, gpu_device)[1] > 0
    xs = [x.view(B, T, H, 64).to(gpu_device) for x in wkv_inputs((B, T), H, seed=T, dtype=dtype).as_tuple()]
    r, w, k, v, a, b = xs
    s0 = wkv_state(B, H).to(gpu_device)
    got_s0 = s0.clone()
    s_out = got_s0 if alias else torch.empty_like(s0)
    y, ck, sa = ops._train_forward(w, r, k, v, a, b, s0=got_s0, s_out=s_out)
    y2, ck2, sa2, s2 = torch.empty_like(y), torch.empty_like(ck), torch.empty_like(sa), torch.empty_like(s0)
    P = _lib.ptr
    _lib.call("rwkv7_wkv_train_forward", _lib.dtype_code(dtype), B, T, H, *(P(x) for x in xs), P(y2), P(s0), P(s2),
              P(ck2), P(sa2), _lib.stream_of(y))
    torch.cuda.synchronize()
    assert close(y, y2, 1e-4, torch.finfo(dtype).eps)
    assert close(sa, sa2, 1e-4) and close(ck, ck2, 1e-4) and close(s_out, s2, 1e-4)


def test_workspace_too_small_runs_unsplit(gpu_device):
    H, T = 4, 512
    print("[case] segmented prefill, small workspace", flush=True)
    ins = [x.to(gpu_device) for x in wkv_inputs((1, T), H, seed=9).as_tuple()]
    need = ops._segment_ws(torch.bfloat16, 1, H, T, T, 0, gpu_device)[1]
    ws = torch.empty(need - 1, dtype=torch.float32, device=gpu_device)
    s1, s2 = wkv_state(1, H).to(gpu_device), wkv_state(1, H).to(gpu_device)
    y1, y2 = torch.empty_like(ins[0]), torch.empty_like(ins[0])
    P = _lib.ptr
    args = (2, 1, T, H * 64, H)
    _lib.call("rwkv7s_forward_ws", *args, P(s1), *(P(x) for x in ins), P(y1), P(ws), need - 1, _lib.stream_of(y1))
    _lib.call("rwkv7s_forward", *args, P(s2), *(P(x) for x in ins), P(y2), _lib.stream_of(y2))
    torch.cuda.synchronize()
    assert torch.equal(y1, y2) and torch.equal(s1, s2)


@pytest.mark.parametrize("lens", [[1], [31, 32, 33], [64, 1, 200], [0, 600, 96], [1500]])
@pytest.mark.parametrize("strong", [False, True])
def test_float32_chunks(gpu_device, lens, strong):
    """The float32 chunked kernel (float32 MFMAs; segmented from a few hundred tokens on) against the float64
    recurrence: 64-term float32 sums carried over the sequence, 2e-6 of the largest magnitude."""
    print(f"[case] float32 prefill lens={lens} strong={strong}", flush=True)
    H, total, n = 4, sum(lens), len(lens)
    ins = [x.to(gpu_device) for x in wkv_inputs((total,), H, seed=total, dtype=torch.float32).as_tuple()]
    if strong:
        ins[1][total // 2, 70] = 1.0
        ins[1][total - 1, 3] = 0.5
    cu = torch.tensor(cu_seqlens_of(lens), dtype=torch.int32, device=gpu_device)
    pool0 = wkv_state(n, H).to(gpu_device)
    pool = pool0.clone()
    y = ops.wkv7_prefill(pool, None, cu, *ins)
    torch.cuda.synchronize()
    for i in range(n):
        lo, hi = cu_seqlens_of(lens)[i], cu_seqlens_of(lens)[i + 1]
        if lo == hi:
            assert torch.equal(pool[i], pool0[i])
            continue
        one = [x[None, lo:hi].double().cpu() for x in ins]
        y64, s64 = ow.wkv7_rowwise(*one, state=pool0[i][None].double().cpu())
        assert close(y[lo:hi], y64[0], 2e-6) and close(pool[i], s64[0], 2e-6)
