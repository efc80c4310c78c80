"""Workspace bounds of the chunked SSD passes — CPU only.

The adjoint scan writes one adjoint per run of R chunks of each head into the
backward workspace, the pipelined and pair chunk kernels read them back, and
every backward workgroup writes a dA partial there; the walking kernels write
and read one map per segment of a head's chunks.  A slot computed past the
end of the workspace is an out-of-bounds write on the GPU (the pair mode's
first run did exactly that: its scan spaced each head's slots nC apart where
the workspace holds ceil(nC / R)).  These tests ask the library for the
largest workspace byte its kernels touch (rr_ssd_workspace_extent: the grids
walked with the kernels' own workgroup decode and slot arithmetic) and check
it against the size the library asks callers for (rr_ssd_workspace_bytes; what
the backward runs against rr_ssd_bwd_workspace_bytes), for BASELINE config 4,
ragged even chunk counts in pair mode, the other modes' shapes, and a sweep over
heads and chunks for the walks.
"""
import pytest

from mlx_recurrence_amd import _lib

BF16 = 1
ALIGN = 256   # every workspace part starts 256-byte aligned

SHAPES = [
    # (B, L, H, Dh, N) at seg 32, bf16, a per-head A (the chunked kernels)
    (8, 4096, 80, 64, 128),    # walks both ways (pass 1's size: pair mode, nC 128)
    (4, 64, 80, 64, 128),      # pair mode, nC 2
    (4, 192, 80, 64, 64),      # walks (pass 1's size: pair mode, nC 6)
    (1, 320, 320, 32, 128),    # pair mode, nC 10, Dh 32
    (5, 1088, 64, 64, 64),     # walks (pass 1's size: pair mode, nC 34)
    (4, 160, 80, 64, 128),     # walks (pass 1's size: nC 5, per-chunk adjoints from the scan)
    (4, 96, 80, 64, 128),      # nC 3 (odd): per-chunk adjoints from the scan
    (2, 1056, 4, 64, 64),      # nC 33, few heads: aggregate + adjoint-pass kernels
    (3, 512, 12, 64, 16),      # sum mode
    (3, 512, 12, 64, 64),      # per-chunk mode, wide state, few heads
    (2, 128, 3, 128, 64),      # wide direct mode (nC 4), Dh 128
    (3, 512, 12, 128, 64),     # wide direct mode: the reference's published shape
    (2, 256, 6, 64, 128),      # Dh 64 N 128, short heads: pipelined
    (4, 512, 16, 128, 64),     # Dh 128, 1024 chunk workgroups: per-chunk mode
    (96, 512, 12, 64, 16),     # SSD c1 shape at B 96: per-chunk with the scan
    (1, 2944, 12, 64, 64),     # walks, many segments
    (2, 1504, 12, 128, 128),   # walks, an uneven last segment
    (5, 128, 56, 64, 128),     # the backward walks in one segment
]


@pytest.mark.parametrize("B,L,H,Dh,N", SHAPES)
@pytest.mark.parametrize("pass_", [0, 1])
def test_kernels_stay_inside_the_workspace(B, L, H, Dh, N, pass_):
    lib = _lib.load()
    need = int(lib.rr_ssd_workspace_bytes(B, L, H, Dh, N, 32, 0, BF16, pass_))
    ext = _lib.ssd_workspace_extent(B, L, H, Dh, N, 32, 0, BF16, pass_)
    assert ext >= 0
    assert ext <= need, f"kernels touch {ext} bytes of a {need}-byte workspace"
    if pass_ == 1:
        # every part of the backward workspace is used up to its alignment padding
        assert need - ext < ALIGN, (need, ext)


@pytest.mark.parametrize("B,L,H,Dh,N", SHAPES)
def test_the_backward_stays_inside_its_own_workspace(B, L, H, Dh, N):
    need = int(_lib.load().rr_ssd_bwd_workspace_bytes(B, L, H, Dh, N, 32, 0, BF16))
    ext = _lib.ssd_bwd_workspace_extent(B, L, H, Dh, N, 32, 0, BF16)
    assert 0 <= ext <= need < ext + ALIGN, (ext, need)


def test_walks_over_heads_and_chunks():
    """Both walks' slots against what their callers allocate, and the backward's
    size against rr_ssd_workspace_bytes(pass = 1), its documented bound."""
    lib = _lib.load()
    walks = 0
    for Dh, N in [(32, 16), (32, 128), (64, 16), (64, 64), (64, 128), (128, 64), (128, 128)]:
        for H in (1, 7, 12, 24, 50, 96, 300, 640, 1500):
            for nC in (1, 2, 3, 5, 17, 23, 33, 47, 92, 128, 257):
                a = (1, 32 * nC, H, Dh, N, 32, 0, BF16)
                assert 0 <= _lib.ssd_workspace_extent(*a, 0) <= lib.rr_ssd_workspace_bytes(*a, 0), a
                ext, need, most = (lib.rr_ssd_bwd_workspace_extent(*a), lib.rr_ssd_bwd_workspace_bytes(*a),
                                   lib.rr_ssd_workspace_bytes(*a, 1))
                assert need <= most, a
                if ext >= 0:   # (Dh 128 with N 16 runs the fp32-MFMA path)
                    assert ext <= need, a
                walks += need != most
    assert walks > 100


def test_pair_mode_bound_detects_the_old_slot_spacing():
    """The bound is tight enough to catch the pair mode's old slot spacing:
    at config 4 the last head's last adjoint, with slots nC (not nC / 2)
    apart per head, lies past the end of the workspace."""
    B, L, H, Dh, N = 8, 4096, 80, 64, 128
    nC, R = L // 32, 2
    lib = _lib.load()
    need = int(lib.rr_ssd_workspace_bytes(B, L, H, Dh, N, 32, 0, BF16, 1))
    ext = _lib.ssd_workspace_extent(B, L, H, Dh, N, 32, 0, BF16, 1)
    state = Dh * N * 4
    agg_end_now = ext                       # the adjoints are the workspace's last part
    last_slot_now = (B * H - 1) * (nC // R) + nC // R - 1
    last_slot_old = (B * H - 1) * nC + nC // R - 1
    agg_begin = agg_end_now - (last_slot_now + 1) * state
    assert agg_begin >= 0
    assert agg_begin + (last_slot_old + 1) * state > need


def test_extent_for_valu_engine_calls_and_bad_arguments():
    # a dense A_neg [H, N] or fp32 inputs run other kernels: no bound from this walk
    assert _lib.ssd_workspace_extent(3, 512, 12, 64, 16, 32, 1, BF16, 1) == -1
    assert _lib.ssd_workspace_extent(3, 512, 12, 64, 16, 32, 0, 0, 1) == -1   # fp32 inputs
    assert _lib.ssd_workspace_extent(0, 512, 12, 64, 16, 32, 0, BF16, 1) == -1
    assert _lib.ssd_workspace_extent(3, 512, 12, 64, 16, 32, 0, BF16, 2) == -1


def test_wide_direct_mode_workspace_at_the_published_shape():
    """The reference's published shape (B3 L512 H12 Dh128 N64, bf16, a rate per
    head) runs the wide direct mode: one kernel per pass, so the forward needs
    no workspace, and the backward holds the dA partials [B,H,nC,N] and one
    adjoint [Dh,N] per chunk (du's operand rows), each part 256-byte aligned.
    Past 768 chunk workgroups the same state takes the resident forward (no
    workspace) and the pipelined backward (per-chunk decays as well)."""
    lib = _lib.load()
    B, L, H, Dh, N = 3, 512, 12, 128, 64
    nC = L // 32

    def al(nbytes):
        return (nbytes + ALIGN - 1) // ALIGN * ALIGN

    assert int(lib.rr_ssd_workspace_bytes(B, L, H, Dh, N, 32, 0, BF16, 0)) == 0
    assert int(lib.rr_ssd_workspace_bytes(B, L, H, Dh, N, 32, 0, BF16, 1)) == \
        al(B * H * nC * N * 4) + al(B * H * nC * Dh * N * 4)
    assert int(lib.rr_gla_workspace_bytes(B, L, H, Dh, 32, BF16, 0)) == 0
    assert int(lib.rr_gla_workspace_bytes(B, L, H, Dh, 32, BF16, 1)) == al(B * H * nC * Dh * Dh * 4)
    # 5 x 12 x 16 = 960 chunk workgroups
    assert int(lib.rr_ssd_workspace_bytes(5, L, H, Dh, N, 32, 0, BF16, 0)) == 0
    assert int(lib.rr_ssd_workspace_bytes(5, L, H, Dh, N, 32, 0, BF16, 1)) == \
        al(5 * H * nC * 4) + al(5 * H * nC * N * 4) + al(5 * H * nC * Dh * N * 4)


def test_few_short_heads_of_dh_32_run_the_direct_kernel():
    """Dh 32, N 128, 4 chunks: one direct kernel (no workspace) up to 64 heads,
    the walk in two segments (their maps) from there; 5 chunks: the pipelined
    kernels (per-chunk decays) up to 48 heads."""
    lib = _lib.load()

    def fwd(H, nC):
        return int(lib.rr_ssd_workspace_bytes(1, 32 * nC, H, 32, 128, 32, 0, BF16, 0))

    assert fwd(24, 4) == fwd(64, 4) == 0 and fwd(72, 4) > 72 * 32 * 128 * 4
    assert 0 < fwd(48, 5) < 4096 and fwd(56, 5) > 56 * 32 * 128 * 4


def test_states_without_a_per_head_scan_never_take_it():
    """From 320 heads the pipelined and pair modes run per-head scans, which are
    not built for the states that walk there (or run direct, resident or whole
    heads): their workspace is never that of those modes."""
    lib = _lib.load()

    def al(n):
        return (n + 63) // 64 * 64 * 4

    for H in [*range(320, 560), 640, 767, 768, 1024, 4099, 65535]:
        for nC in [*range(1, 36), 64, 129]:
            for Dh, N in [(32, 64), (64, 64), (32, 128), (64, 128), (128, 128)]:
                assert lib.rr_ssd_workspace_bytes(1, 32 * nC, H, Dh, N, 32, 0, BF16, 0) != al(H * nC), (H, nC, Dh, N)
            for Dh in (64, 128):
                assert lib.rr_gla_workspace_bytes(1, 32 * nC, H, Dh, 32, BF16, 0) != al(H * nC), (H, nC, Dh)
            own = lib.rr_ssd_bwd_workspace_bytes(1, 32 * nC, H, 64, 64, 32, 0, BF16)
            for runs in {nC, nC // 2}:
                assert own != al(H * nC) + al(H * runs * 64) + al(H * runs * 64 * 64), (H, nC)
            gla = lib.rr_gla_workspace_bytes(1, 32 * nC, H, 64, 32, BF16, 1)
            assert gla != al(H * nC) + al(H * nC * 64 * 64), (H, nC)
