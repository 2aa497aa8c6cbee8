"""The native decode step (``rwkv7_decode_layers``) against the loop of
``forward_pooled`` it stands for: the same kernels in the same order on the same
operands, so logits and states are equal bit for bit - at row counts of every tile
plan, with rows without a slot, fewer logit rows than rows, and without ln0."""

import pytest
import torch

from rwkvtune_amd import _lib
from rwkvtune_amd.model import RWKV7Config, StatePool, build_model

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def model(gpu_device):
    cfg = RWKV7Config(n_layer=3, n_embd=512, vocab_size=1024, dim_att_lora=32, dim_gate_lora=96, dim_mv_lora=64)
    return build_model(cfg, torch.bfloat16, gpu_device, seed=1)


def step(m, native, tokens, slots, pool0, rows=None):
    pool = StatePool(m.config, pool0.n_slots, m.device)
    for dst, src in ((pool.kv, pool0.kv), (pool.att_x, pool0.att_x), (pool.ffn_x, pool0.ffn_x)):
        dst.copy_(src)
    m.packs()
    keep = m._rows
    m._rows = keep if native else None
    try:
        last = torch.arange(tokens.numel(), dtype=torch.int32, device=m.device)
        out = m.forward_pooled(tokens, slots, last, pool, decode=True, logit_rows=rows)
    finally:
        m._rows = keep
    torch.cuda.synchronize()
    return out, pool


@pytest.mark.parametrize("M", [1, 8, 31, 33, 65, 129, 256])
@pytest.mark.parametrize("skip_ln0", [False, True])
def test_equals_the_layer_loop(model, gpu_device, M, skip_ln0):
    print(f"[case] native decode step M={M} skip_ln0={skip_ln0}", flush=True)
    m = model
    m.blocks[0].skip_ln0 = skip_ln0
    m.invalidate()
    g = torch.Generator(device=gpu_device).manual_seed(M)
    S = M + 3
    pool0 = StatePool(m.config, S, gpu_device)
    for t in (pool0.kv, pool0.att_x, pool0.ffn_x):
        t.copy_(torch.randn(t.shape, generator=g, device=gpu_device) * 0.3)
    tokens = torch.randint(0, 1024, (M,), generator=g, device=gpu_device)
    slots = torch.randperm(S, generator=g, device=gpu_device)[:M].to(torch.int32)
    if M > 8:
        slots[5] = -1
    rows = torch.arange(0, M, 2, dtype=torch.int32, device=gpu_device) if M % 2 else None
    a, pa = step(m, True, tokens, slots, pool0, rows)
    b, pb = step(m, False, tokens, slots, pool0, rows)
    assert a.shape[0] == (M if rows is None else rows.numel())
    assert torch.equal(a, b)
    assert torch.equal(pa.kv, pb.kv) and torch.equal(pa.att_x, pb.att_x) and torch.equal(pa.ffn_x, pb.ffn_x)
    m.blocks[0].skip_ln0 = False
    m.invalidate()


def test_states_of_any_float_type_are_copied(model, gpu_device):
    """forward_with_state copies its input states (here half of them in float64) and leaves them alone."""
    print("[case] native decode step, states", flush=True)
    m = model
    st = m.init_state(4)
    g = torch.Generator(device=gpu_device).manual_seed(2)
    for s in st:
        for k in s:
            s[k] = torch.randn(s[k].shape, generator=g, device=gpu_device) * 0.2
    st64 = [{k: (v.double() if i % 2 else v) for i, (k, v) in enumerate(s.items())} for s in st]
    keep = [{k: v.clone() for k, v in s.items()} for s in st64]
    tok = torch.tensor([[3], [5], [7], [9]], device=gpu_device)
    a, na = m.forward_with_state(tok, st)
    b, nb = m.forward_with_state(tok, st64)
    assert torch.equal(a, b) and all(torch.equal(x[k], y[k]) for x, y in zip(na, nb) for k in x)
    assert all(torch.equal(x[k], y[k]) for x, y in zip(keep, st64) for k in x)
    with pytest.raises(ValueError):
        m.forward_with_state(tok, st[:2])


def test_arguments_are_checked(model, gpu_device):
    print("[case] native decode step, arguments", flush=True)
    m = model
    m.packs()
    lib = _lib.load()
    assert lib.rwkv7_decode_layers_scratch(0, 512, 2048, 3, m._rows) == -1
    assert lib.rwkv7_decode_layers_ws_floats(4, 512, 2048, 3, None) == -1
    with pytest.raises(ValueError, match="scratch"):
        _lib.call("rwkv7_decode_layers", 4, 512, 2048, 3, m._rows, *[None] * 2, 1024, *[None] * 5, 4, *[None] * 3, 4,
                  None, None, 0, None, 0, None)


def test_uniform_layout(model, gpu_device):
    """Slots, last rows and offsets of B sequences of T rows."""
    for B, T in ((1, 1), (3, 1), (1, 5), (4, 7)):
        slot, last, cu, seq = model._meta_uniform(B, T, gpu_device)
        want = torch.full((B * T,), -1, dtype=torch.int32)
        want[0::T] = torch.arange(T - 1, B * T, T, dtype=torch.int32)
        assert all(t.dtype == torch.int32 and t.is_contiguous() for t in (slot, last, cu, seq))
        assert slot.tolist() == [i // T for i in range(B * T)] and last.cpu().tolist() == want.tolist()
        assert cu.tolist() == list(range(0, (B + 1) * T, T)) and seq.tolist() == list(range(B))
