'''Chord inputs whose rows lie off 16-byte boundaries: copied, not refused.'''
import pytest
import torch

from motif.ops.chord_attention import _aligned


def _shifted(t, n=1):
    '''t's values, contiguous, n elements into a buffer.'''
    buf = torch.zeros(t.numel() + n, dtype=t.dtype, device=t.device)
    v = buf[n:].view(t.shape)
    v.copy_(t)
    return v


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16, torch.float32])
def test_aligned_copies(dtype):
    t = torch.randn(2, 3, 5, 64).to(dtype)
    for x in (_shifted(t), t[:, :, :1].as_strided((2, 3, 1, 64), (960, 320, 67, 1)),
              t[:1].as_strided((1, 3, 5, 64), (3, 320, 64, 1))):
        a = _aligned(x)
        assert torch.equal(a, x) and a.data_ptr() % 16 == 0
        assert all(s * a.element_size() % 16 == 0 for s in a.stride()[:-1])
    assert _aligned(t).data_ptr() == t.data_ptr()


@pytest.mark.gpu
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float32])
@pytest.mark.parametrize('L,S', [(40, 40), (1, 70)])
def test_forward_at_odd_offsets(dtype, L, S):
    import motif.ops as ops
    from test_gpu_chord_wide import DEV, _inputs
    q, k, v, par = _inputs(2, 4, 2, L, S, 64, dtype, 3)
    log_n = torch.log(torch.arange(S - L + 1, S + 1, dtype=torch.float32))[None].expand(2, L).contiguous()
    rest = [p.to(DEV) for p in par] + [log_n.to(DEV)]
    ref = ops.apply_chord_attention(q.to(DEV), k.to(DEV), v.to(DEV), *rest)
    got = ops.apply_chord_attention(*(_shifted(t.to(DEV)) for t in (q, k, v)), *rest)
    assert torch.equal(got, ref)


@pytest.mark.gpu
def test_backward_at_odd_offsets():
    from motif.ops import apply_chord_attention
    from test_gpu_chord_bwd import DEV, _inputs
    x = _inputs(1, 4, 2, 50, 50, 3)
    log_n = torch.log(torch.arange(1, 51, dtype=torch.float32, device=DEV))[None].contiguous()

    def grads(lay):
        ts = [lay(t.to(DEV)).requires_grad_() for t in x[:3]] + [t.to(DEV).requires_grad_() for t in x[3:7]]
        return torch.autograd.grad(apply_chord_attention(*ts, log_n), ts, lay(x[7].to(DEV)))
    assert all(torch.equal(a, b) for a, b in zip(grads(_shifted), grads(lambda t: t)))
