"""GPU parity at BASELINE config 4's full workload (MI355X only).

ssd_scan forward + backward at B=8, L=4096, H=80, Dh=64, N=128, bf16 inputs,
fp32 state, seg=32: 128 checkpoint intervals per head.  At this shape both
passes walk a head's chunks (final_fwd.hip with checkpoints, walk_bwd.hip in two
segments per head, the second one's adjoint map first).

The inputs are drawn on the device (config 0's distributions) and rounded to
bf16 there.  Every (batch, head) is an independent scan, so the float64 oracle
(oracle/recurrence_oracle.py, reference ssd.py:203-268) is run on whole heads:
all 8 batch rows of heads 0, 41 and 79, which makes dA[h] (summed over the
batch) complete for those heads.  The loss is sum(y * W) with W ~ N(0,1) (the
reference's parity loss, _chassis.py:171-175).

Bars: outputs kept in fp32 (y, final state, dA) 1e-5 normalised error (the
fp32 bar of the north star); bf16 gradients 2e-2.
"""
from __future__ import annotations

import math

import numpy as np
import pytest
import torch

from oracle import recurrence_oracle as orc
from tests.gpu_util import rel_err

import mlx_recurrence_amd as mr

pytestmark = pytest.mark.gpu

B, L, H, Dh, N, SEG = 8, 4096, 80, 64, 128, 32
HEADS = (0, 41, 79)
FP32_BAR = 1e-5
BF16_BAR = 2e-2


@pytest.fixture(scope="module")
def c4_run():
    """One forward + backward at the full config-4 shape; returns the
    per-head slices (float64, CPU) of inputs and results."""
    print(f"[case] ssd_c4 B={B} L={L} H={H} Dh={Dh} N={N} seg={SEG} bf16", flush=True)
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(4)
    bf = torch.bfloat16
    u = torch.randn((B, L, H, Dh), generator=g, device=dev).to(bf)
    delta = (torch.randn((B, L, H), generator=g, device=dev).abs() * 0.1 + 0.01).to(bf)
    Bm = torch.randn((B, L, H, N), generator=g, device=dev).to(bf)
    Cm = torch.randn((B, L, H, N), generator=g, device=dev).to(bf)
    A = -torch.exp(torch.rand((H,), generator=g, device=dev) * math.log(16.0))
    W = torch.randn((B, L, H, Dh), generator=g, device=dev)
    xs = [t.requires_grad_(True) for t in (u, delta, Bm, Cm, A)]
    y, fs = mr.ssd_scan_with_state(xs[0], xs[1], xs[2], xs[3], xs[4][:, None].expand(H, N), seg=SEG)
    y.backward(W)
    torch.cuda.synchronize()
    hs = list(HEADS)

    def cpu(t, axis):
        return t.detach().index_select(axis, torch.tensor(hs, device=dev)).double().cpu().numpy()

    out = dict(
        u=cpu(u, 2), delta=cpu(delta, 2), Bm=cpu(Bm, 2), Cm=cpu(Cm, 2), A=cpu(A, 0), W=cpu(W, 2),
        y=cpu(y, 2), fs=cpu(fs, 1), du=cpu(xs[0].grad, 2), dd=cpu(xs[1].grad, 2), dB=cpu(xs[2].grad, 2),
        dC=cpu(xs[3].grad, 2), dA=cpu(xs[4].grad, 0),
    )
    assert xs[0].grad.dtype == bf and y.dtype == torch.float32 and fs.shape == (B, H, Dh, N)
    del u, delta, Bm, Cm, A, W, xs, y, fs
    torch.cuda.empty_cache()
    return out


@pytest.mark.parametrize("j", range(len(HEADS)), ids=[f"head{h}" for h in HEADS])
def test_ssd_c4_head_parity(c4_run, j):
    r = c4_run
    sl = (slice(None), slice(None), slice(j, j + 1))
    u, dl, Bm, Cm = r["u"][sl], r["delta"][:, :, j:j + 1], r["Bm"][sl], r["Cm"][sl]
    A = np.repeat(r["A"][j:j + 1, None], N, axis=1)            # [1, N], one rate per head
    print(f"[case] ssd_c4 oracle head {HEADS[j]}", flush=True)
    y_o, fs_o = orc.ssd_forward(u, dl, Bm, Cm, A)
    du_o, dd_o, dB_o, dC_o, dA_o, _ = orc.ssd_backward(r["W"][sl], u, dl, Bm, Cm, A)
    errs = {
        "y": rel_err(r["y"][sl], y_o), "final": rel_err(r["fs"][:, j:j + 1], fs_o),
        "grad_A": rel_err(r["dA"][j:j + 1], dA_o.sum(1)),
        "grad_u": rel_err(r["du"][sl], du_o), "grad_delta": rel_err(r["dd"][:, :, j:j + 1], dd_o),
        "grad_B": rel_err(r["dB"][sl], dB_o), "grad_C": rel_err(r["dC"][sl], dC_o),
    }
    print(f"ssd_c4 head {HEADS[j]}: " + " ".join(f"{k}={v:.2e}" for k, v in errs.items()), flush=True)
    for k in ("y", "final", "grad_A"):
        assert errs[k] < FP32_BAR, (k, errs)
    for k in ("grad_u", "grad_delta", "grad_B", "grad_C"):
        assert errs[k] < BF16_BAR, (k, errs)
