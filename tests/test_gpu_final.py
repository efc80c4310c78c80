"""The walking forward (final_fwd.hip: bf16, one decay rate per head for SSD; in
calls without a gradient it keeps no checkpoints) against the float64 oracle
and against the general path, at the edges of its chunks and segments (MI355X
only).

Bar: it works to fp32 accuracy (three-term bf16 splits, fp32 accumulation), so
outputs are held to the fp32 bar, 1e-5 of the largest value."""
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


def _ssd(B, L, H, Dh, N, seed):
    rng = np.random.default_rng(seed)
    return [to_dev(rng.standard_normal((B, L, H, Dh)), BF16),
            to_dev(np.abs(rng.standard_normal((B, L, H))) * 0.1 + 0.01, BF16),
            to_dev(rng.standard_normal((B, L, H, N)), BF16), to_dev(rng.standard_normal((B, L, H, N)), BF16),
            to_dev(-np.exp(rng.uniform(0, np.log(16), H)), F32)], to_dev(rng.standard_normal((B, H, Dh, N)), F32)


def _gla(B, L, H, Dh, seed):
    rng = np.random.default_rng(seed)
    g = 1 / (1 + np.exp(-(rng.standard_normal((B, L, H)) + 2)))
    g[:, L // 2] *= -1          # either sign
    g[:, L // 3] = 0            # a reset
    return ([to_dev(rng.standard_normal((B, L, H, Dh)) / np.sqrt(Dh), BF16) for _ in range(3)] + [to_dev(g, BF16)],
            to_dev(rng.standard_normal((B, H, Dh, Dh)), F32))


# (B, L, H, Dh, N, seg): one step, a chunk less one, a chunk plus one, odd tails,
# every Dh and N, several segments (1000 and 2040 steps of few heads), T = 32
SSD = [(1, 1, 2, 32, 16, 1), (2, 31, 1, 64, 128, 31), (1, 33, 3, 128, 32, 11), (2, 40, 5, 32, 64, 8),
       (1, 100, 3, 64, 64, 4), (2, 1000, 3, 64, 16, 8), (1, 2040, 2, 32, 128, 8), (1, 520, 2, 128, 128, 8),
       (1, 72, 2, 128, 16, 24), (1, 77, 2, 32, 32, 7), (3, 544, 8, 64, 128, 32), (1, 768, 24, 64, 32, 32)]
GLA = [(1, 1, 2, 64, 1), (2, 31, 1, 32, 31), (1, 33, 3, 128, 11), (1, 1000, 2, 64, 8), (2, 520, 1, 128, 8),
       (1, 100, 3, 32, 20), (1, 544, 24, 64, 32)]


@pytest.mark.parametrize("h0", [False, True])
@pytest.mark.parametrize("B,L,H,Dh,N,seg", SSD)
def test_ssd_final(B, L, H, Dh, N, seg, h0):
    print(f"[case] ssd final B={B} L={L} H={H} Dh={Dh} N={N} seg={seg} h0={h0}", flush=True)
    assert _lib.ssd_final_workspace(B, L, H, Dh, N, seg, 0, BF16) >= 0
    ins, st = _ssd(B, L, H, Dh, N, L + Dh)
    y, fs = mr.ssd_scan_with_state(*ins, seg=seg, initial_state=st if h0 else None)
    ref = [rounded(t) for t in ins]
    ref[4] = np.repeat(ref[4][:, None], N, axis=1)
    y_o, fs_o = orc.ssd_forward(*ref, rounded(st) if h0 else None)
    rep = {}
    assert y.shape == (B, L, H, Dh) and fs.shape == (B, H, Dh, N)
    check("y", y, y_o, TOL[F32], rep)
    check("final", fs, fs_o, TOL[F32], rep)
    print(rep, flush=True)


@pytest.mark.parametrize("h0", [False, True])
@pytest.mark.parametrize("B,L,H,Dh,seg", GLA)
def test_gla_final(B, L, H, Dh, seg, h0):
    print(f"[case] gla final B={B} L={L} H={H} Dh={Dh} seg={seg} h0={h0}", flush=True)
    assert _lib.gla_final_workspace(B, L, H, Dh, seg, BF16) >= 0
    ins, st = _gla(B, L, H, Dh, L + Dh)
    y, fs = mr.gla_scan_with_state(*ins, seg=seg, initial_state=st if h0 else None)
    y_o, fs_o = orc.gla_forward(*[rounded(t) for t in ins], rounded(st) if h0 else None)
    rep = {}
    check("y", y, y_o, TOL[F32], rep)
    check("final", fs, fs_o, TOL[F32], rep)
    print(rep, flush=True)


# training calls whose forward walks (17 chunks: several segments, an odd one
# last; 64 chunks of more heads: fewer segments), every Dh with its widest N
WALKS = [("ssd", 1, 544, 24, 64, 64), ("ssd", 2, 544, 12, 64, 128), ("ssd", 1, 576, 24, 32, 128),
         ("ssd", 1, 544, 24, 128, 128), ("ssd", 1, 1024, 24, 64, 16), ("gla", 1, 544, 24, 64, 64),
         ("gla", 2, 544, 12, 128, 128), ("gla", 3, 2048, 24, 32, 32), ("ssd", 1, 128, 24, 64, 128)]


@pytest.mark.parametrize("kind,B,L,H,Dh,N", WALKS)
def test_walking_training_forward(kind, B, L, H, Dh, N):
    """y and the checkpoints (the state after every chunk) of rr_ssd_fwd and
    rr_gla_fwd where they walk."""
    print(f"[case] walk {kind} B={B} L={L} H={H} Dh={Dh} N={N}", flush=True)
    ins, st = _ssd(B, L, H, Dh, N, 3) if kind == "ssd" else _gla(B, L, H, Dh, 3)
    y = torch.empty((B, L, H, Dh), device=st.device)
    ckpt = torch.full((B, H, L // 32, Dh, N), float("nan"), device=st.device)
    if kind == "ssd":
        ws = _lib.ssd_workspace(B, L, H, Dh, N, 32, 0, BF16, 0, st.device)
        _lib.ssd_fwd(*ins, 0, st, 32, y, ckpt, ws)
        ref = [rounded(t) for t in ins]
        ref[4] = np.repeat(ref[4][:, None], N, axis=1)
        fwd = orc.ssd_forward
    else:
        ws = _lib.gla_workspace(B, L, H, Dh, 32, BF16, 0, st.device)
        _lib.gla_fwd(*ins, st, 32, y, ckpt, ws)
        ref = [rounded(t) for t in ins]
        fwd = orc.gla_forward
    rep = {}
    y_o, fs_o = fwd(*ref, rounded(st))
    check("y", y, y_o, TOL[F32], rep)
    for c in (0, 1, L // 64, L // 32 - 1):
        cut = [r[:, :32 * (c + 1)] if r.ndim >= 3 else r for r in ref]
        _, h = fwd(*cut, rounded(st))
        got = ckpt[:, :, c] if kind == "ssd" else ckpt[:, :, c].transpose(-1, -2)
        check(f"ckpt {c}", got, h, TOL[F32], rep)
    assert not torch.isnan(ckpt).any()
    print(rep, flush=True)


def test_forms_agree_with_the_recording_path():
    """Every form the call accepts (strided and misaligned inputs, the three
    forms of A_neg, mixed dtypes) gives what the path with checkpoints gives;
    calls it does not cover go there."""
    B, L, H, Dh, N, seg = 2, 72, 3, 64, 32, 8
    ins, st = _ssd(B, L, H, Dh, N, 5)
    u, d, Bm, Cm, A = ins
    pad = torch.empty(u.numel() + 1, dtype=BF16, device=u.device)[1:]
    odd = pad.copy_(u.flatten()).view_as(u)                                   # 2-byte aligned
    strided = u.transpose(1, 2).contiguous().transpose(1, 2)
    stt = st.transpose(-1, -2).contiguous().transpose(-1, -2)
    forms = [(u, d, Bm, Cm, A), (odd, d, Bm, Cm, A), (strided, d, Bm, Cm, A[:, None].expand(H, N)),
             (u, d, Bm.float(), Cm, A), (u, d, Bm, Cm, A[:, None].expand(H, N).contiguous())]
    for k, f in enumerate(forms):
        print(f"[case] form {k}", flush=True)
        y, fs = mr.ssd_scan_with_state(*f, seg=seg, initial_state=stt)
        yr, fr = mr.ssd_scan_with_state(f[0].detach().requires_grad_(True), *f[1:], seg=seg, initial_state=stt)
        for got, want in ((y, yr), (fs, fr)):
            assert got.dtype == want.dtype and got.shape == want.shape and not got.requires_grad
            assert (got - want).abs().max() <= 1e-5 * want.abs().max(), k
    assert _lib.ssd_final_workspace(B, L, H, Dh, N, seg, 1, BF16) == -1     # dense A
    assert _lib.ssd_final_workspace(B, L, H, Dh, N, seg, 0, F32) == -1
    assert _lib.ssd_final_workspace(B, L, H, 96, N, seg, 0, BF16) == -1


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_non_finite_input_stays_causal(bad):
    """A non-finite u, B or C at one step leaves every earlier step as it was."""
    B, L, H, Dh, N, s = 1, 72, 2, 64, 128, 41
    ins, st = _ssd(B, L, H, Dh, N, 9)
    clean, _ = mr.ssd_scan_with_state(*ins, seg=8, initial_state=st)
    for k in (0, 2, 3):
        xs = [t.clone() for t in ins]
        xs[k][0, s, 1, 5] = bad
        y, _ = mr.ssd_scan_with_state(*xs, seg=8, initial_state=st)
        assert torch.equal(y[:, :s], clean[:, :s]) and torch.equal(y[:, :, 0], clean[:, :, 0]), k
        assert not torch.isfinite(y[0, s, 1]).all(), k


def _same(got, want, tol):
    """Infinities and NaN where the recurrence has them; the finite values within tol."""
    got = got.detach().double().cpu().numpy()
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isinf(got), np.isinf(want)) and np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    ok = np.isfinite(want)
    assert np.abs(got[ok] - want[ok]).max(initial=0) <= tol * np.abs(want[ok]).max(initial=0)


# one and several segments, a whole number of chunks (walking, with and without checkpoints)
@pytest.mark.parametrize("kind,B,L,H,N,seg,grad", [("ssd", 1, 72, 2, 128, 8, False), ("ssd", 1, 1000, 2, 16, 8, False),
                                                   ("ssd", 1, 544, 24, 64, 32, False), ("ssd", 1, 544, 24, 64, 32, True),
                                                   ("gla", 1, 1000, 2, 64, 8, False), ("gla", 1, 544, 24, 64, 32, True)])
def test_infinities_follow_the_recurrence(kind, B, L, H, N, seg, grad):
    """One infinite input, or one in the initial state: y and the final state have
    infinities and NaN exactly where the recurrence has them."""
    ins, st = _ssd(B, L, H, 64, N, 9) if kind == "ssd" else _gla(B, L, H, 64, 9)
    fn, ref = ((mr.ssd_scan_with_state, orc.ssd_forward) if kind == "ssd" else
               (mr.gla_scan_with_state, orc.gla_forward))
    if kind == "gla":
        ins[3] = ins[3].abs().clamp(min=0.5)   # no resets: zero times infinity
    s = L // 2 + 5
    for k in range(5):   # u, delta, B, C (q, k, v, gates), initial state
        xs, x0 = [t.clone() for t in ins], st.clone()
        if k < 4:
            xs[k][(0, s, 1, 5)[:xs[k].ndim]] = float("inf")
        else:
            x0[0, 1, 5, 7] = float("inf")
        print(f"[case] inf {kind} L={L} N={N} seg={seg} grad={grad} input {k}", flush=True)
        r = [rounded(t) for t in xs]
        if kind == "ssd":
            r[4] = np.repeat(r[4][:, None], N, axis=1)
        with np.errstate(all="ignore"):
            y_o, fs_o = ref(*r, rounded(x0))
        if grad:
            xs[0].requires_grad_(True)
        y, fs = fn(*xs, seg=seg, initial_state=x0)
        _same(y, y_o, TOL[F32])
        _same(fs, fs_o, TOL[F32])


def test_growing_gates_over_an_empty_start():
    """Gates above 1 whose product over a segment overflows, over steps that add
    nothing to a zero state: no infinity times zero."""
    B, L, H, Dh = 1, 1000, 2, 64
    (q, k, v, g), _ = _gla(B, L, H, Dh, 4)
    g[:, :640], v[:, :640] = 6.0, 0.0
    g[:, 640:] = g[:, 640:].abs().clamp(min=0.5)
    y, fs = mr.gla_scan_with_state(q, k, v, g, seg=8)
    y_o, fs_o = orc.gla_forward(*[rounded(t) for t in (q, k, v, g)])
    assert np.isfinite(y_o).all()
    _same(y, y_o, TOL[F32])
    _same(fs, fs_o, TOL[F32])
