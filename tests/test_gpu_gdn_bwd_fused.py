'''The one-call backward of the chunk rule (motif_gdn_chunk_bwd) against the float64 torch form:
chunk edges, both value widths, caller layouts its row loads take and do not take, output
gradients that are broadcast, missing state gradients, mixed input types.'''
import pytest
import torch

from motif.ops import chunk_gated_delta_rule
from motif.ops.autograd_path import gdn_chunk_torch
from support import gdn_inputs

pytestmark = pytest.mark.gpu
DEV = 'cuda'


def _ref(x, S0, do, dS):
    ts = [t.double().requires_grad_() for t in x]
    s0 = S0.double().requires_grad_()
    o, S = gdn_chunk_torch(*ts, s0)
    return torch.autograd.grad([o, S], [*ts, s0], [do.double(), dS.double()])


def _bar(x):
    '''fp32: the rounding of the cumulative decays, 2^-24 max |gamma| of a chunk, enters every
    term (twice: e^gamma and e^-gamma), and sums of up to 128 products of order-one terms
    add 2^-24 sqrt(128) each along a chain of eight products.  bf16 gradients: half an ulp,
    2^-9, on top.'''
    g = x[4].double()
    pad = -g.shape[2] % 64
    gam = torch.nn.functional.pad(g, (0, pad)).reshape(*g.shape[:2], -1, 64).sum(-1).abs().max().item()
    return (2 * gam + 8 * 128 ** 0.5) * 2 ** -24 + (2 ** -8 if x[0].dtype == torch.bfloat16 else 0.0)


def _check(x, S0, do, dS, lay=lambda t: t.to(DEV)):
    ref = _ref(x, S0, do, dS)
    ts = [lay(t).requires_grad_() for t in x]
    s0 = S0.to(DEV).requires_grad_()
    o, S = chunk_gated_delta_rule(*ts, s0)
    got = torch.autograd.grad([o, S], [*ts, s0], [lay(do.to(o.dtype)), dS.to(DEV)])
    for name, a, r, t in zip('qkvbgS', got, ref, [*ts, s0]):
        assert a.dtype == t.dtype and a.shape == t.shape, name
        err = ((a.double().cpu() - r).norm() / r.norm().clamp_min(1e-30)).item()
        assert err < _bar(x), (name, err)


def _case(B, H, L, dv, dtype=torch.float32):
    x = gdn_inputs(B, H, L, 64, dv, seed=L + dv, dtype=dtype)
    g = torch.Generator().manual_seed(L)
    do = torch.randn(B, H, L, dv, generator=g).to(dtype)
    return x, 0.1 * torch.randn(B, H, 64, dv, generator=g), do, 0.1 * torch.randn(B, H, 64, dv, generator=g)


@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
@pytest.mark.parametrize('B,H,L,dv', [(1, 2, 2, 64), (2, 1, 63, 128), (1, 3, 64, 64), (2, 2, 65, 128), (1, 2, 321, 64)])
def test_edges(B, H, L, dv, dtype):
    _check(*_case(B, H, L, dv, dtype))


@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
@pytest.mark.parametrize('shift', [0, 1, 4])
def test_layouts(dtype, shift):
    '''[B, T, H, D] storage inside wider rows, at an element offset that keeps (4) or breaks
    (1) the four-element row alignment.'''
    def lay(t):
        p = t.transpose(1, 2)
        if p.dim() == 3:
            return p.to(DEV).contiguous().transpose(1, 2)
        wide = torch.zeros(*p.shape[:3], p.shape[3] + 8, dtype=p.dtype, device=DEV)
        v = wide[..., shift:shift + p.shape[3]]
        v.copy_(p)
        return v.transpose(1, 2).detach()
    _check(*_case(2, 3, 130, 128, dtype), lay=lay)


def test_broadcast_output_gradient_and_no_state():
    x, _, _, _ = _case(1, 2, 100, 64)
    ts = [t.double().requires_grad_() for t in x]
    ref = torch.autograd.grad(gdn_chunk_torch(*ts)[0].sum(), ts)
    ts = [t.to(DEV).requires_grad_() for t in x]
    got = torch.autograd.grad(chunk_gated_delta_rule(*ts)[0].sum(), ts)  # (an expanded gradient: stride 0)
    for a, r in zip(got, ref):
        assert ((a.double().cpu() - r).norm() / r.norm()).item() < _bar(x)


def test_mixed_types():
    x, S0, do, dS = _case(1, 2, 70, 128)
    x[0], x[2] = x[0].bfloat16(), x[2].bfloat16()
    ref = _ref(x, S0, do.bfloat16(), dS)
    ts = [t.to(DEV).requires_grad_() for t in x]
    o, S = chunk_gated_delta_rule(*ts, S0.to(DEV))
    got = torch.autograd.grad([o, S], ts, [do.bfloat16().to(DEV), dS.to(DEV)])
    for a, r, t in zip(got, ref, ts):
        assert a.dtype == t.dtype
        assert ((a.double().cpu() - r).norm() / r.norm()).item() < _bar(x) + 2 ** -8


@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
def test_empty_sequence_passes_the_state_gradient(dtype):
    x, S0, do, dS = _case(2, 3, 0, 64, dtype)
    ts = [t.to(DEV).requires_grad_() for t in x]
    s0 = S0.to(DEV).requires_grad_()
    o, S = chunk_gated_delta_rule(*ts, s0)
    assert o.shape == do.shape and torch.equal(S, s0)
    got = torch.autograd.grad([o, S], [*ts, s0], [do.to(DEV), dS.to(DEV)])
    assert all(a.shape == t.shape for a, t in zip(got, [*ts, s0]))
    assert torch.equal(got[-1].cpu(), dS)


@pytest.mark.parametrize('transpose', [False, True])
@pytest.mark.parametrize('dk,dv,shift', [(64, 128, 0), (64, 16, 1), (32, 48, 3), (16, 32, 0)])
@pytest.mark.parametrize('N', [0, 1, 2, 3, 4, 5, 9])
def test_operator_scan_depths(N, dk, dv, shift, transpose):
    '''Chain lengths around the scan's load depth, operands and records at any element
    address.  Bar: a step rounds dk products and sums of order one, 2^-24 (dk / 4 + 8), and
    the contraction (|A| <= 1/2) keeps the sum over the steps below twice one step's.'''
    from motif.ops.gdn_grad import opscan
    g = torch.Generator().manual_seed(dk + N)

    def rand(*shape):
        n = torch.Size(shape).numel()
        return torch.randn(n + shift, generator=g).to(DEV)[shift:].view(shape)
    A = 0.5 * torch.linalg.qr(torch.randn(2, 3, max(N, 1), dk, dk, generator=g))[0][:, :, :N].to(DEV)
    Q, S0 = rand(2, 3, N, dk, dv), rand(2, 3, dk, dv)
    P, S = opscan(A, Q, S0, reverse=transpose, transpose=transpose)
    ref = S0.double().cpu()
    for n in (reversed(range(N)) if transpose else range(N)):
        assert (P[:, :, n].double().cpu() - ref).abs().max() <= 2 ** -23 * (dk / 4 + 8) * ref.abs().max()
        M = A[:, :, n].double().cpu()
        ref = (M.transpose(-1, -2) if transpose else M) @ ref + Q[:, :, n].double().cpu()
    assert (S.double().cpu() - ref).abs().max() <= 2 ** -23 * (dk / 4 + 8) * ref.abs().max()


def test_more_batch_rows_than_a_grid_dimension():
    '''65540 one-step rows: the rows on both sides of the launch limit as in a call of their own.'''
    g = torch.Generator(device=DEV).manual_seed(3)
    r = lambda *s: torch.randn(65540, 1, 1, *s, generator=g, device=DEV)  # noqa: E731
    x = [r(64), r(64), r(64), torch.sigmoid(r()), -torch.rand(65540, 1, 1, generator=g, device=DEV)]
    do = r(64)

    def grads(rows):
        ts = [t[rows].requires_grad_() for t in x]
        return torch.autograd.grad(chunk_gated_delta_rule(*ts)[0], ts, do[rows])
    whole = grads(slice(None))
    for rows in (slice(0, 3), slice(65533, 65540)):
        assert all(torch.equal(a[rows], b) for a, b in zip(whole, grads(rows)))
