'''The Chord backward at the edges of its 32-row tiles, 6-tile chunks and 128-row blocks, with the
output gradient in the [B, L, H, D] storage a layer hands back, inside a wider row and broadcast
over heads; same reference and bars as tests/test_gpu_chord_bwd.py.'''
import math

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


@pytest.mark.parametrize('L,S', [(1, 2), (33, 33), (70, 100)])
def test_output_gradient_broadcast_over_rows(L, S):
    '''One gradient row for every query (row stride 0, what a sum over the queries hands back):
    the rows past L of the last tile share its elements and still count as zeros.'''
    from motif.ops import apply_chord_attention
    x = _inputs(2, 4, 2, L, S, 7 + L)
    log_n = torch.log(torch.arange(S - L + 1, S + 1, dtype=torch.float32) + 1)[None].expand(2, L).contiguous()
    row = x[7][:, :, :1]
    _, ref = _grads_torch64(*x[:7], log_n, S - L, row.expand(2, 4, L, 64))
    ts = [t.to(DEV).requires_grad_(True) for t in x[:7]]
    dout = row.to(DEV).expand(2, 4, L, 64)
    assert dout.stride(2) == 0 or L == 1
    got = torch.autograd.grad(apply_chord_attention(*ts, log_n.to(DEV)), ts, dout)
    for name, a, r in zip(('dq', 'dk', 'dv'), got[:3], ref[:3]):
        _close(a.cpu(), r, f'{name} L={L}')


def test_one_row_of_any_stride():
    '''A single query and key row whose stride is past the staging offsets (never used).  One
    key: dq and dk are zero up to the rounding of two 64-term dots of products below 16,
    2 * 64 * 16 * 2^-24; dv is a bf16 rounding.'''
    from motif.ops import apply_chord_attention
    x = _inputs(1, 2, 1, 1, 1, 3)
    log_n = torch.full((1, 1), 0.7)
    _, ref = _grads_torch64(*x[:7], log_n, 0, x[7])
    far = lambda t: t.to(DEV).as_strided(t.shape, (t.stride(0), t.stride(1), 1 << 26, 1))
    ts = [far(t).requires_grad_(True) for t in x[:3]] + [t.to(DEV).requires_grad_(True) for t in x[3:7]]
    got = torch.autograd.grad(apply_chord_attention(*ts, log_n.to(DEV)), ts, far(x[7]))
    for name, a, r in zip(('dq', 'dk', 'dv'), got[:3], ref[:3]):
        assert (a.double().cpu() - r).abs().max() <= 2 ** -8 * r.abs().max() + 2 ** -13, name


@pytest.mark.parametrize('L', [70, 640])
def test_dq_operand_rounding(L):
    '''dQ is the bf16 of the fp32 sum of bf16(s c dZ) times K, one chunk of keys or several, with P
    from the forward's own log-sum-exp (of its 16-bit P) and Delta from its 16-bit output.  P
    carries a few 2^-20 from the exponential, so a share of 2^-20 / 2^-9 of the operands rounds
    the other way (2^-8 each, of a sum of many: below 1e-4), and with that a share of 1e-4 / 2^-8
    of the results (2^-8 each: 6e-4).  With the factor s c outside the rounding the distance is
    that of two independent roundings, 3.4e-3.'''
    from motif.ops import apply_chord_attention
    from motif.ops.chord_attention import _launch
    q, k, v, alpha, beta, mu, ssmax, dout = _inputs(1, 2, 2, L, L, 11 + L)
    log_n = torch.log(torch.arange(1, L + 1, dtype=torch.float32))[None].contiguous()
    ts = [t.to(DEV).requires_grad_(True) for t in (q, k, v, alpha, beta, mu, ssmax)]
    out = apply_chord_attention(*ts, log_n.to(DEV))
    dq = torch.autograd.grad(out, ts[0], dout.to(DEV))[0].double().cpu()
    lse = torch.empty(1, 2, L, device=DEV)
    with torch.no_grad():
        _launch(*ts, log_n.to(DEV), 0, 0.125, 1e-5, torch.empty_like(out), lse)

    col = lambda t: t.double().view(1, 2, 1, 1)  # noqa: E731
    d = torch.arange(L)[None].double() - torch.arange(L)[:, None].double()
    c = col(ssmax) * log_n.double().view(1, 1, L, 1)
    bias = -col(alpha) * ((d - col(mu)).abs() + 1e-5) ** col(beta)
    z = ((q.double() @ k.double().transpose(-1, -2)) * 0.125 + bias) * c
    P = torch.exp2(z.masked_fill(d > 0, float('-inf')) * math.log2(math.e) - lse.double().cpu()[..., None])
    delta = (dout.double() * out.detach().double().cpu()).sum(-1, keepdim=True)
    dz = P * (dout.double() @ v.double().transpose(-1, -2) - delta)
    want = ((dz * c * 0.125).bfloat16().double() @ k.double()).bfloat16().double()
    assert ((dq - want).norm() / want.norm()).item() < 1e-3


@pytest.mark.parametrize('form', ['far', 'backwards', 'workspace'])
def test_entry_takes_any_row_stride_and_workspace(form):
    '''motif_chord_bwd itself on rows 2^25 elements apart (0.3 GB each), rows that run backwards,
    and a workspace off 16-byte boundaries: the bits of the plain call.'''
    from motif.ops import _lib
    from motif.ops.chord_attention import _launch
    q, k, v, alpha, beta, mu, ssmax, dout = (t.to(DEV) for t in _inputs(1, 1, 1, 5, 5, 9))
    log_n = torch.log(torch.arange(1, 6, dtype=torch.float32, device=DEV))[None].contiguous()
    out, lse = torch.empty_like(q), torch.empty(1, 1, 5, device=DEV)
    with torch.no_grad():
        _launch(q, k, v, alpha, beta, mu, ssmax, log_n, 0, 0.125, 1e-5, out, lse)

    def arg(t):
        if form == 'far':
            buf = torch.zeros((4 << 25) + 64, dtype=t.dtype, device=DEV)
            rows = buf.as_strided(t.shape, (0, 0, 1 << 25, 1))
            rows.copy_(t)
            return buf, [buf.data_ptr(), 0, 0, 1 << 25]
        if form == 'backwards':
            buf = t.flip(2).contiguous()
            return buf, [buf[0, 0, 4].data_ptr(), 0, 0, -64]
        return t, _lib.t4(t)

    def call(args, shift):
        grads = [torch.empty_like(t) for t in (q, k, v)]
        par = torch.empty(4, 1, device=DEV)
        n = int(_lib.lib().motif_chord_bwd_workspace_bytes(1, 1, 1, 5, 5, 0))
        ws = torch.empty(n + 16, dtype=torch.uint8, device=DEV)
        a = [x for _, t in args[:3] for x in t] + _lib.t4(out) + args[3][1]
        rc = _lib.lib().motif_chord_bwd(
            *a, lse.data_ptr(), *(t.data_ptr() for t in (alpha, beta, mu, ssmax, log_n)), 5, 1,
            *(x for t in grads for x in _lib.t4(t)), par.data_ptr(), 1, 1, 1, 5, 5, 64, 0, 0.125, 1e-5,
            ws.data_ptr() + shift, n, _lib.chord_dtype_code(q.dtype), _lib.stream_ptr(q.device))
        _lib.check(rc, 'motif_chord_bwd')
        return [*grads, par]
    plain = call([(t, _lib.t4(t)) for t in (q, k, v, dout)], 0)
    got = call([arg(t) for t in (q, k, v, dout)], 4 if form == 'workspace' else 0)
    assert all(torch.equal(a, b) for a, b in zip(got, plain))
