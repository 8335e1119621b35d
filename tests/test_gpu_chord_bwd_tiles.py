'''The Chord backward at the edges of its 32-row tiles, 6-tile chunks and 128-row blocks, with the
output gradient in the [B, L, H, D] storage a layer hands back, inside a wider row and broadcast
over heads; same reference and bars as tests/test_gpu_chord_bwd.py.'''
import pytest
import torch

from test_gpu_chord_bwd import DEV, _close, _grads_torch64, _inputs

pytestmark = pytest.mark.gpu


def _layouts(dout):
    B, H, L, D = dout.shape
    yield dout.transpose(1, 2).contiguous().to(DEV).transpose(1, 2)
    wide = torch.zeros(B, L, H, D + 8, dtype=dout.dtype, device=DEV)
    wide[..., 8:] = dout.transpose(1, 2).to(DEV)
    yield wide[..., 8:].transpose(1, 2)


@pytest.mark.parametrize('B,H,Hkv,L,S', [(1, 2, 1, 31, 31), (1, 4, 2, 33, 161), (2, 2, 2, 191, 191), (1, 2, 1, 193, 193),
                                         (1, 3, 3, 257, 400)])
def test_tile_and_chunk_edges(B, H, Hkv, L, S):
    from motif.ops import apply_chord_attention
    x = _inputs(B, H, Hkv, L, S, L + S)
    log_n = torch.log(torch.arange(S - L + 1, S + 1, dtype=torch.float32))[None].expand(B, L).contiguous()
    _, ref = _grads_torch64(*x[:7], log_n, S - L, x[7])
    for dout in _layouts(x[7]):
        ts = [t.to(DEV).requires_grad_(True) for t in x[:7]]
        out = apply_chord_attention(*ts, log_n.to(DEV))
        got = torch.autograd.grad(out, ts, dout)
        for name, a, r in zip(('dq', 'dk', 'dv'), got[:3], ref[:3]):
            _close(a.cpu(), r, f'{name} L={L} S={S}')
        for a, r in zip(got[3:], ref[3:]):
            assert ((a.double().cpu() - r).norm() / r.norm()).item() < 3e-2


def test_broadcast_output_gradient():
    '''One gradient for every head (stride 0): read as it is.'''
    from motif.ops import apply_chord_attention
    x = _inputs(1, 4, 2, 70, 70, 5)
    log_n = torch.log(torch.arange(1, 71, dtype=torch.float32))[None].contiguous()
    one = x[7][:, :1]
    _, ref = _grads_torch64(*x[:7], log_n, 0, one.expand(1, 4, 70, 64))
    ts = [t.to(DEV).requires_grad_(True) for t in x[:7]]
    got = torch.autograd.grad(apply_chord_attention(*ts, log_n.to(DEV)), ts, one.to(DEV).expand(1, 4, 70, 64))
    for name, a, r in zip(('dq', 'dk', 'dv'), got[:3], ref[:3]):
        _close(a.cpu(), r, name)
