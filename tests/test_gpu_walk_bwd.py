"""The walking backward (walk_bwd.hip) against the float64 oracle at the least
chunk counts that take it, with an initial state and a final-state cotangent:
one to many segments, an uneven last one, every Dh x N; GLA with gates of either
sign and resets (MI355X only).  Bars: those of tests/gpu_util.py (bf16
gradients: storage rounding; fp32 outputs 1e-4)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import mlx_recurrence_amd as mr
from mlx_recurrence_amd import _lib
from oracle import recurrence_oracle as orc
from tests.gpu_util import TOL, check, rounded, to_dev

pytestmark = pytest.mark.gpu
BF16, F32 = torch.bfloat16, torch.float32

CASES = [  # kind, B, L, H, Dh, N
    ("ssd", 1, 2944, 12, 64, 64),      # 92 chunks of 12 heads: many segments
    ("ssd", 2, 1504, 12, 64, 128),     # 47 chunks, an uneven last segment
    ("ssd", 1, 1504, 24, 128, 64),
    ("ssd", 5, 128, 56, 64, 128),      # 4 chunks of 280 heads: one segment
    ("ssd", 3, 64, 184, 128, 128),     # 2 chunks
    ("gla", 1, 2944, 12, 64, 64),
    ("gla", 4, 160, 55, 64, 64),
    ("gla", 1, 1504, 24, 128, 128),
]


@pytest.mark.parametrize("kind,B,L,H,Dh,N", CASES)
def test_walk_bwd(kind, B, L, H, Dh, N):
    print(f"[case] walk_bwd {kind} B={B} L={L} H={H} Dh={Dh} N={N}", flush=True)
    rng = np.random.default_rng(L + N)
    h0 = to_dev(rng.standard_normal((B, H, Dh, N)), F32, True)
    W = rng.standard_normal((B, L, H, Dh)).astype(np.float32).astype(np.float64)
    Wf = rng.standard_normal((B, H, Dh, N)).astype(np.float32).astype(np.float64)
    if kind == "ssd":
        xs = [to_dev(rng.standard_normal((B, L, H, Dh)), BF16, True),
              to_dev(np.abs(rng.standard_normal((B, L, H))) * 0.1 + 0.01, BF16, True),
              to_dev(rng.standard_normal((B, L, H, N)), BF16, True), to_dev(rng.standard_normal((B, L, H, N)), BF16, True),
              to_dev(-np.exp(rng.uniform(0, np.log(16), H)), F32, True)]
        y, fs = mr.ssd_scan_with_state(*xs, initial_state=h0)
        ref = [rounded(t) for t in xs]
        ref[4] = np.repeat(ref[4][:, None], N, axis=1)
        grads = list(orc.ssd_backward(W, *ref, rounded(h0), Wf))
        grads[4] = grads[4].sum(1)
        names = ["u", "delta", "B", "C", "A"]
    else:
        g = 1 / (1 + np.exp(-(rng.standard_normal((B, L, H)) + 2)))
        g[:, L // 2] *= -1
        g[:, 5:7] *= -1
        g[:, L // 3] = 0
        xs = [to_dev(rng.standard_normal((B, L, H, Dh)) / np.sqrt(Dh), BF16, True) for _ in range(3)]
        xs.append(to_dev(g, BF16, True))
        y, fs = mr.gla_scan_with_state(*xs, initial_state=h0)
        grads = list(orc.gla_backward(W, *[rounded(t) for t in xs], rounded(h0), Wf))
        names = ["q", "k", "v", "g"]
    ((y * to_dev(W, F32)).sum() + (fs * to_dev(Wf, F32)).sum()).backward()
    rep = {}
    for name, t, want in zip(names + ["h0"], xs + [h0], grads):
        check("grad_" + name, t.grad, want, TOL[BF16], rep)
    print(rep, flush=True)


def test_growing_gates_after_the_last_cotangent():
    """Gates above 1 whose product over a segment overflows, after the last step
    that the loss sees: the adjoint of a zero cotangent is zero."""
    B, L, H, Dh = 1, 2944, 12, 64
    rng = np.random.default_rng(7)
    x = [rng.standard_normal((B, L, H, Dh)) / 8 for _ in range(3)]
    g = 1 / (1 + np.exp(-(rng.standard_normal((B, L, H)) + 2)))
    W = rng.standard_normal((B, L, H, Dh)).astype(np.float32).astype(np.float64)
    g[:, 600] = 0
    g[:, 601:], x[1][:, 601:], x[2][:, 600:], W[:, 600:] = 6.0, 0, 0, 0
    xs = [to_dev(t, BF16, True) for t in (*x, g)]
    y, _ = mr.gla_scan_with_state(*xs)
    (y * to_dev(W, F32)).sum().backward()
    grads = list(orc.gla_backward(W, *[rounded(t) for t in xs], None, None))
    rep = {}
    for name, t, want in zip(["q", "k", "v", "g"], xs, grads):
        assert np.isfinite(want).all()
        check("grad_" + name, t.grad, want, TOL[BF16], rep)
    print(rep, flush=True)


@pytest.mark.parametrize("kind,B,L,H,Dh,N", [("ssd", 5, 128, 56, 64, 128), ("ssd", 1, 2944, 12, 64, 64),
                                             ("ssd", 1, 1504, 24, 128, 128), ("gla", 1, 1504, 24, 128, 128)])
def test_walks_write_inside_their_buffers(kind, B, L, H, Dh, N):
    """Forward and backward with workspaces of exactly the stated size and outputs
    of exactly their shapes, each followed by a byte pattern that must stay: one
    segment (no maps) and several."""
    print(f"[case] walk guards {kind} B={B} L={L} H={H} Dh={Dh} N={N}", flush=True)
    rng = np.random.default_rng(5)
    guard, keep = 1 << 20, []

    def buf(shape, dtype):
        n = int(np.prod(shape)) * torch.empty(0, dtype=dtype).element_size()
        b = torch.full((n + guard,), 0x5A, dtype=torch.uint8, device="cuda")
        keep.append(b[n:])
        return b[:n].view(dtype).view(shape)

    def ws(n):
        assert n % 4 == 0
        return buf((n,), torch.uint8) if n else None

    lib, dt = _lib.load(), _lib.DTYPE_CODE[BF16]
    dy = to_dev(rng.standard_normal((B, L, H, Dh)), F32)
    st, df = (to_dev(rng.standard_normal((B, H, Dh, N)), F32) for _ in range(2))
    y, ckpt, dh0 = buf((B, L, H, Dh), F32), buf((B, H, L // 32, Dh, N), F32), buf((B, H, Dh, N), F32)
    if kind == "ssd":
        size = (B, L, H, Dh, N, 32, 0, dt)
        need = lib.rr_ssd_bwd_workspace_bytes(*size)
        assert need < lib.rr_ssd_workspace_bytes(*size, 1)   # the backward walks
        xs = [to_dev(rng.standard_normal((B, L, H, Dh)), BF16), to_dev(np.abs(rng.standard_normal((B, L, H))) * 0.1, BF16),
              to_dev(rng.standard_normal((B, L, H, N)), BF16), to_dev(rng.standard_normal((B, L, H, N)), BF16),
              to_dev(-np.exp(rng.uniform(0, 2, H)), F32)]
        grads = [buf(x.shape, BF16) for x in xs[:4]] + [buf((H, N), F32)]
        _lib.ssd_fwd(*xs, 0, st, 32, y, ckpt, ws(lib.rr_ssd_workspace_bytes(*size, 0)))
        _lib.ssd_bwd(dy, df, *xs, 0, st, ckpt, 32, *grads, dh0, ws(need))
    else:
        size = (B, L, H, Dh, 32, dt)
        xs = [to_dev(rng.standard_normal((B, L, H, Dh)) / 8, BF16) for _ in range(3)]
        xs.append(to_dev(1 / (1 + np.exp(-(rng.standard_normal((B, L, H)) + 2))), BF16))
        grads = [buf(x.shape, BF16) for x in xs]
        _lib.gla_fwd(*xs, st, 32, y, ckpt, ws(lib.rr_gla_workspace_bytes(*size, 0)))
        _lib.gla_bwd(dy, df, *xs, st, ckpt, 32, *grads, dh0, ws(lib.rr_gla_workspace_bytes(*size, 1)))
    torch.cuda.synchronize()
    assert all(bool((g == 0x5A).all()) for g in keep)
    for t in (y, ckpt, dh0, *grads):
        assert bool(torch.isfinite(t.float()).all())
