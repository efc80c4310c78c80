"""Size limits of the SSD and GLA entry points — CPU only (the size queries and
the refusals before any launch).

A call is refused with and without a gradient alike: the forward without
checkpoints takes nothing that rr_ssd_fwd / rr_gla_fwd refuse."""
import ctypes

import pytest

from mlx_recurrence_amd import _lib

BF16 = 1
PTR = ctypes.c_void_p(16)   # never dereferenced: validation fails first

BEYOND = [(65536, 8, 1, "B and H must be <= 65535"), (1, 8, 65536, "B and H must be <= 65535"),
          (65535, 32776, 1, "B*L too large")]


@pytest.mark.parametrize("B,L,H,text", BEYOND)
def test_no_gradient_calls_are_refused_like_the_others(B, L, H, text):
    lib = _lib.load()
    assert lib.rr_ssd_final_workspace_bytes(B, L, H, 64, 16, 8, 0, BF16) == -1
    assert lib.rr_gla_final_workspace_bytes(B, L, H, 64, 8, BF16) == -1
    for rc in (lib.rr_ssd_final_fwd(PTR, PTR, PTR, PTR, PTR, 0, BF16, B, L, H, 64, 16, 8, None, PTR, PTR, None, 0, None),
               lib.rr_ssd_fwd(PTR, PTR, PTR, PTR, PTR, 0, BF16, B, L, H, 64, 16, 8, None, PTR, PTR, None, 0, None),
               lib.rr_gla_final_fwd(PTR, PTR, PTR, PTR, BF16, B, L, H, 64, 8, None, PTR, PTR, None, 0, None),
               lib.rr_gla_fwd(PTR, PTR, PTR, PTR, BF16, B, L, H, 64, 8, None, PTR, PTR, None, 0, None)):
        assert rc == _lib.RR_EUNSUPPORTED and text.encode() in lib.rr_last_error()
    assert lib.rr_ssd_final_workspace_bytes(65535, 8, 1, 64, 16, 8, 0, BF16) == 0
    assert lib.rr_gla_final_workspace_bytes(1, 8, 65535, 64, 8, BF16) == 0


@pytest.mark.parametrize("Dh,heads", [(128, 1 << 23), (64, 1 << 24), (32, 1 << 25)])
def test_walks_stay_below_the_launch_limit(Dh, heads):
    """HIP launches fewer than 2^32 threads, and a walk uses 4 Dh (backward:
    at most 512) of them per head in a 1-D grid: more heads run elsewhere."""
    lib = _lib.load()
    H = 32768
    B = heads // H
    assert lib.rr_ssd_final_workspace_bytes(B, 1, H, Dh, 16, 1, 0, BF16) == -1
    assert lib.rr_ssd_final_workspace_bytes(B, 1, H - 1, Dh, 16, 1, 0, BF16) >= 0
    assert lib.rr_gla_final_workspace_bytes(B, 1, H, Dh, 1, BF16) == -1
    assert lib.rr_gla_final_workspace_bytes(B, 1, H - 1, Dh, 1, BF16) >= 0


def test_walking_backward_stays_below_the_launch_limit():
    lib = _lib.load()
    for B, walks in ((256, False), (255, True)):   # 2^23 heads of two chunks
        H = 32768
        own = lib.rr_ssd_bwd_workspace_bytes(B, 64, H, 128, 128, 32, 0, BF16)
        assert (own < lib.rr_ssd_workspace_bytes(B, 64, H, 128, 128, 32, 0, BF16, 1)) == walks
