'''The Chord backward's chunk plan, read from the workspace it asks for (no GPU): fp32 partial
planes only where cutting the causal loops pays, none where the launch fills the chip by itself.'''
import pytest

from motif.ops import _lib


def _planes(B, H, Hkv, L, S):
    '''(dQ, dK / dV) partial planes, and the bytes that every plan needs.'''
    q_start = S - L
    got = _lib.lib().motif_chord_bwd_workspace_bytes(B, H, Hkv, L, S, q_start) - 16  # (room to align an odd base)
    al = lambda n: -(-n // 256) * 256  # noqa: E731
    nqb = -(-L // 128)
    hits = []
    for nq in range(1, 9):
        for nkv in range(0, 9):
            n = al(16 * B * H * L) + al(16 * nq * B * nqb * H) + (al(256 * nq * B * H * L) if nq > 1 else 0)
            if n + 2 * al(256 * nkv * H * B * S) == got:
                hits.append((nq, nkv))
    assert len(hits) == 1, (got, hits)
    return hits[0]


@pytest.mark.parametrize('B,H,L', [(8, 12, 256), (12, 12, 256), (16, 12, 256), (12, 12, 384), (12, 12, 512),
                                   (16, 12, 512), (32, 12, 512), (32, 16, 384), (64, 8, 256)])
def test_full_launches_are_not_cut(B, H, L):
    assert _planes(B, H, H, L, L) == (1, 0)
    assert _planes(B, H, H // 4, L, L) == (1, 1)


@pytest.mark.parametrize('B,H,L,S', [(1, 12, 512, 512), (1, 12, 1024, 1024), (2, 12, 2048, 2048), (1, 12, 4096, 4096),
                                     (1, 8, 64, 4096)])
def test_short_launches_are_cut(B, H, L, S):
    nq, nkv = _planes(B, H, H, L, S)
    assert nq > 1 and (nkv > 1 or L < 512)


def test_one_tile_and_no_queries():
    assert _planes(1, 1, 1, 1, 1) == (1, 0)
    assert _lib.lib().motif_chord_bwd_workspace_bytes(1, 2, 1, 0, 10, 0) > 0
