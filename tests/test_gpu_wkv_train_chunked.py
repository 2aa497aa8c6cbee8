"""The chunked training backward (``rwkv7_wkv_train_backward_chunked``) against the
float64 oracle, where its tiles, segments and fallbacks begin and end.

* T around the 16-token checkpoints and the 32-token chunks; few (sequence, head)
  units, so that the sequence is cut into one segment per chunk, and 256 of them,
  where one block walks the whole sequence;
* a chunk below the matrix form's log-decay floor (token-serial inside the kernel),
  also with its segment neighbours in matrix form;
* initial state and final-state gradient, the start state given or recovered from
  the first checkpoint; unaligned tensors (token-serial kernel).

Tolerances.  The matrix form's float32 products and sums leave up to ~1e-6 of a
tensor's largest magnitude; recovering a start state divides by the decay of up to
16 tokens (>= 0.577 each here: a factor <= 7e3 on 6e-8).  float32 gradients: 1e-5
of the largest magnitude, 2e-3 with a recovered start.  16-bit gradients: one ulp
of the value (rounding, and a tie the other way) plus 2e-3 of the largest
magnitude for the hi / lo operand parts and the recovered start.
"""

import pytest
import torch

from oracle import wkv7_train as otr
from rwkvtune_amd import operators as ops

pytestmark = pytest.mark.gpu


def make(B, T, H, dtype, seed, strong=()):
    g = torch.Generator().manual_seed(seed)
    shp = (B, T, H, 64)
    r, k, v, dy = (torch.randn(shp, generator=g) for _ in range(4))
    w = torch.rand(shp, generator=g) * 5.4 - 6.0
    for t in strong:
        w[0, t, 0, 7] = 1.0  # log-decay -e
    kk = torch.nn.functional.normalize(torch.randn(shp, generator=g), dim=-1)
    b = kk * torch.rand(shp, generator=g)
    s0 = torch.randn(B, H, 64, 64, generator=g) * 0.1
    ds = torch.randn(B, H, 64, 64, generator=g) * 0.1
    return [x.to(dtype) for x in (r, w, k, v, -kk, b)], dy.to(dtype), s0, ds


def check(name, got, ref, dtype, frac, scale=0.0):
    ref = ref.double()
    err = (got.double().cpu() - ref).abs()
    ulp = 0.0 if dtype == torch.float32 else torch.finfo(dtype).eps
    bound = ulp * ref.abs() + frac * max(float(ref.abs().max()), scale)
    assert bool((err <= bound).all()), (name, float((err - bound).max()), float(ref.abs().max()))


def run(dev, B, T, H, dtype, state, known, seed, strong=(), shift=False):
    xs, dy, s0, ds = make(B, T, H, dtype, seed, strong)
    r, w, k, v, a, b = (x.double() for x in xs)
    s0o = s0.double() if state else None
    y_o, sa_o, ck_o, _ = otr.train_forward(r, w, k, v, a, b, s0=s0o)
    want = otr.train_backward(r, w, k, v, a, b, dy.double(), ck_o, sa_o, ds_in=ds.double() if state else None)

    def put(x):
        x = x.to(dev)
        if not shift:
            return x.contiguous()
        buf = torch.empty(x.numel() + 1, dtype=x.dtype, device=dev)
        buf[1:] = x.reshape(-1)
        return buf[1:].view(x.shape)

    rd, wd, kd, vd, ad, bd = (put(x) for x in xs)
    s0d = s0.to(dev) if state else None
    y, ck, sa = ops._train_forward(wd, rd, kd, vd, ad, bd, s0=s0d)
    dw, dr, dk, dv, da, db, ds0 = ops._train_backward(
        wd, rd, kd, vd, ad, bd, put(dy), ck, sa, ds_in=ds.to(dev) if state else None, want_ds0=True,
        s0=s0d if known else None, start_known=known)
    torch.cuda.synchronize()
    frac = 1e-5 if dtype == torch.float32 and known and not strong else 2e-3
    for name, got, ref in zip(("dr", "dw", "dk", "dv", "da", "db"), (dr, dw, dk, dv, da, db), want):
        assert got.dtype == dtype
        # dw is a difference of suffix sums whose terms are as large as lw r dr (their rounding stays where
        # they cancel: one token from a zero state has dw = 0)
        scale = float((w.exp() * r * want[0]).abs().max()) if name == "dw" else 0.0
        check(name, got, ref, dtype, frac, scale)
    check("ds0", ds0, want[6], torch.float32, 1e-5)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T", [1, 15, 16, 17, 31, 32, 33, 96, 113])
@pytest.mark.parametrize("state,known", [(True, True), (True, False), (False, True)])
def test_lengths(gpu_device, dtype, T, state, known):
    print(f"[case] chunked backward {dtype} T={T} state={state} known={known}", flush=True)
    run(gpu_device, 2, T, 3, dtype, state, known, seed=T)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("strong", [(5,), (40,), (20, 70), (95,)])
def test_strong_decay_chunk(gpu_device, dtype, strong):
    print(f"[case] chunked backward {dtype} strong decay at {strong}", flush=True)
    run(gpu_device, 2, 100, 2, dtype, True, True, seed=7, strong=strong)


@pytest.mark.parametrize("B,H", [(8, 32), (4, 33), (5, 24)])
def test_many_units(gpu_device, B, H):
    """256 units (one block per unit over the whole sequence), 132 and 120 (one and two segments)."""
    print(f"[case] chunked backward B={B} H={H}", flush=True)
    run(gpu_device, B, 70, H, torch.bfloat16, True, True, seed=B, strong=(40,))


def test_unaligned_tensors_run_token_by_token(gpu_device):
    print("[case] chunked backward unaligned", flush=True)
    run(gpu_device, 1, 37, 2, torch.bfloat16, True, True, seed=3, shift=True)


@pytest.mark.parametrize("special", [float("inf"), float("nan"), -float("inf")])
def test_non_finite_decay_input(gpu_device, special):
    """w = +inf is decay 0, NaN is NaN from its token on; neither may reach other sequences, and
    w = -inf is decay 1."""
    print(f"[case] chunked backward w={special}", flush=True)
    xs, dy, s0, ds = make(2, 64, 2, torch.bfloat16, 11)
    xs[1][0, 40, 0, 3] = special
    dev = [x.to(gpu_device) for x in xs]
    r, w, k, v, a, b = dev
    y, ck, sa = ops._train_forward(w, r, k, v, a, b)
    out = ops._train_backward(w, r, k, v, a, b, dy.to(gpu_device), ck, sa, want_ds0=True, start_known=True)
    clean = [x[1:].contiguous() for x in dev]
    r1, w1, k1, v1, a1, b1 = clean
    y1, ck1, sa1 = ops._train_forward(w1, r1, k1, v1, a1, b1)
    ref = ops._train_backward(w1, r1, k1, v1, a1, b1, dy[1:].to(gpu_device).contiguous(), ck1, sa1, want_ds0=True,
                              start_known=True)
    torch.cuda.synchronize()
    for got, want in zip(out, ref):
        assert torch.isfinite(got[1:]).all() and torch.allclose(got[1:].float(), want.float(), rtol=1e-2, atol=1e-2)
    if special == -float("inf"):
        assert all(bool(torch.isfinite(x).all()) for x in out)
