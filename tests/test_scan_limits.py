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
