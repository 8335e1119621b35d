'''The fp32 chunk rule on the matrix instructions (csrc/gdn_f32.hip) against the float64
oracle: chunk edges, every head shape of its dispatch and the one past it, carried states,
unaligned and transposed rows, packed sequences.'''
import pytest
import torch

import motif.ops as ops
from oracle import gdn as ogdn
from support import gdn_inputs

pytestmark = pytest.mark.gpu
DEV = 'cuda'


def _bar(g):
    '''Relative bound: a decay e^{gamma_C - gamma} carries the rounding of the cumulative sums
    gamma, up to max |gamma| 2^-24 each; eight more 2^-23 for the sums of 64 products and the
    triangular solve.'''
    n = -(-g.shape[2] // 64) * 64
    gam = torch.nn.functional.pad(g, (0, n - g.shape[2])).reshape(*g.shape[:2], -1, 64).sum(-1).abs().max().item()
    return (8 + gam) * 2 ** -23


def _rel(x, y):
    return ((x.double().cpu() - y).norm() / y.norm()).item()


@pytest.mark.parametrize('dk,dv', [(64, 64), (64, 128), (64, 32), (32, 96), (32, 64), (32, 160)])
@pytest.mark.parametrize('B,T', [(1, 1), (2, 63), (1, 64), (1, 65), (2, 200), (1, 641)])
def test_chunk_f32_edges(B, T, dk, dv):
    x = gdn_inputs(B, 3, T, dk, dv, seed=T + dv)
    g = torch.Generator().manual_seed(T)
    S = 0.1 * torch.randn(B, 3, dk, dv, generator=g) if T % 2 else None
    ro, rS = ogdn.chunked(*(t.double() for t in x), None if S is None else S.double(), 64)
    o, S1 = ops.chunk_gated_delta_rule(*(t.to(DEV) for t in x), None if S is None else S.to(DEV))
    assert _rel(o, ro) < _bar(x[4]) and _rel(S1, rS) < _bar(x[4])


def test_chunk_f32_strides():
    '''[B, T, H, D] storage at an odd element offset: rows off 16-byte boundaries.'''
    x = gdn_inputs(2, 3, 130, 64, 96, seed=5)
    ro, rS = ogdn.chunked(*(t.double() for t in x), None, 64)

    def shifted(t):
        buf = torch.empty(t.numel() + 1, device=DEV)
        perm = t.transpose(1, 2)
        v = buf[1:].view(perm.shape)
        v.copy_(perm)
        return v.transpose(1, 2)
    o, S = ops.chunk_gated_delta_rule(*(shifted(t) for t in x))
    assert _rel(o, ro) < _bar(x[4]) and _rel(S, rS) < _bar(x[4])


def test_chunk_f32_packed():
    lens = [1, 64, 0, 130, 63]
    cu = torch.tensor([0, 1, 65, 65, 195, 258], dtype=torch.int32)
    x = gdn_inputs(1, 2, sum(lens), 64, 128, seed=9)
    S0 = 0.1 * torch.randn(5, 2, 64, 128, generator=torch.Generator().manual_seed(1))
    ro, rS = ogdn.chunked_varlen(*(t.double() for t in x), cu, S0.double(), 64)
    o, S = ops.chunk_gated_delta_rule_varlen(*(t.to(DEV) for t in x), cu.to(DEV), S0.to(DEV))
    assert _rel(o, ro) < _bar(x[4]) and _rel(S, rS) < _bar(x[4])
