'''The fp32-arithmetic Chord prefill (csrc/chord_wide.hip) against the float64 oracle: edges of
its 32-query blocks and of the 8 x 32-key round of its waves, every type and head dim it serves,
continued and clipped key ranges, signs of ssmax and scale, strided destinations.'''
import pytest
import torch

import motif.ops as ops
from oracle import chord as ochord

pytestmark = pytest.mark.gpu
DEV = 'cuda'
# fp32: logits of up to ~60 log2 units carry 60 2^-24 into exp2, twice for the bias and the
# product, and the sums a little more; 16-bit results: half an ulp of the type (2^-9 / 2^-12)
# on top
BAR = {torch.float32: 1e-5, torch.float16: 2 ** -11, torch.bfloat16: 2 ** -8}


def _inputs(B, H, Hkv, L, S, D, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(B, H, L, D, generator=g).to(dtype)
    k = torch.randn(B, Hkv, S, D, generator=g).to(dtype)
    v = torch.randn(B, Hkv, S, D, generator=g).to(dtype)
    par = [torch.exp(0.3 * torch.randn(H, generator=g)), 0.2 * torch.randn(H, generator=g),
           0.2 * torch.randn(H, generator=g), 1 + 0.1 * torch.randn(H, generator=g)]
    return q, k, v, par


def _check(q, k, v, par, q_start=None, scale=None, out=None):
    B, H, L, D = q.shape
    qs = k.shape[2] - L if q_start is None else q_start
    ln = ochord.log_n_table(qs, L).float()[None].expand(B, L).contiguous()
    ref = ochord.chord_attention(q, k, v, *par, ln, qs, scale)
    got = ops.apply_chord_attention(q.to(DEV), k.to(DEV), v.to(DEV), *(p.to(DEV) for p in par), ln.to(DEV),
                                    q_start=qs, softmax_scale=scale, out=out)
    err = ((got.double().cpu() - ref).norm() / ref.norm()).item()
    assert err < BAR[q.dtype], err


@pytest.mark.parametrize('L,S', [(9, 9), (31, 31), (32, 32), (33, 97), (64, 256), (65, 257), (257, 300), (600, 600)])
@pytest.mark.parametrize('dtype', [torch.float32, torch.float16])
def test_wide_sizes(L, S, dtype):
    _check(*_inputs(2, 4, 2, L, S, 64, dtype, L + S))


@pytest.mark.parametrize('D', [16, 32, 128, 48])
@pytest.mark.parametrize('dtype', [torch.float32, torch.float16, torch.bfloat16])
def test_wide_head_dims(D, dtype):
    _check(*_inputs(1, 3, 1, 70, 300, D, dtype, D))


@pytest.mark.parametrize('scale', [0.2, -0.2, 0.0])
def test_wide_signs(scale):
    q, k, v, par = _inputs(1, 4, 4, 40, 40, 64, torch.float32, 3)
    par[3] = par[3] * torch.tensor([1., -1., 1., -1.])
    _check(q, k, v, par, scale=scale)


def test_wide_clipped_keys_and_strided_out():
    '''Queries past the last key (they see every key), keys past the last query, an output
    in [B, L, H, D] storage.'''
    x = _inputs(2, 3, 3, 50, 41, 64, torch.float32, 7)
    out = torch.empty(2, 50, 3, 64, device=DEV).transpose(1, 2)
    _check(*x, q_start=20, out=out)
    _check(*_inputs(1, 3, 3, 50, 400, 64, torch.float32, 8), q_start=100)


@pytest.mark.parametrize('dtype', [torch.float32, torch.float16])
@pytest.mark.parametrize('B,H,Hkv,L,S,D', [(64, 16, 1, 2, 512, 64), (64, 8, 2, 3, 300, 64), (48, 16, 1, 1, 600, 32),
                                           (64, 16, 1, 2, 40, 128)])
def test_short_queries_in_large_batches(B, H, Hkv, L, S, D, dtype):
    '''Sizes around the rule that leaves short query blocks of many heads per kv head to the
    vector kernel.'''
    _check(*_inputs(B, H, Hkv, L, S, D, dtype, S))


@pytest.mark.parametrize('stride', [(1 << 24) - 8, 1 << 24])
def test_far_rows(stride):
    '''Key rows on both sides of the stride that the flash kernel's 32-bit tile offsets hold (past
    it: the vector kernel); 20 rows span 0.64 GB.'''
    q, k, v, par = _inputs(1, 2, 1, 20, 20, 64, torch.float16, 4)
    buf = torch.zeros(19 * stride + 64, dtype=torch.float16, device=DEV)
    far = buf.as_strided((1, 1, 20, 64), (0, 0, stride, 1))
    far.copy_(k)
    ln = ochord.log_n_table(0, 20).float()[None].contiguous()
    ref = ochord.chord_attention(q, k, v, *par, ln, 0, None)
    got = ops.apply_chord_attention(q.to(DEV), far, v.to(DEV), *(p.to(DEV) for p in par), ln.to(DEV))
    assert ((got.double().cpu() - ref).norm() / ref.norm()).item() < BAR[torch.float16]


def test_far_single_rows():
    '''The stride of a single row does not count: a query and a key row whose stride lies past the
    tile offsets.'''
    far = lambda t: t.to(DEV).as_strided(t.shape, (t.stride(0), t.stride(1), 1 << 26, 1))  # noqa: E731
    q, k, v, par = _inputs(2, 16, 1, 1, 30, 64, torch.float32, 6)
    ln = ochord.log_n_table(29, 1).float()[None].expand(2, 1).contiguous()
    ref = ochord.chord_attention(q, k, v, *par, ln, 29, None)
    got = ops.apply_chord_attention(far(q), k.to(DEV), v.to(DEV), *(p.to(DEV) for p in par), ln.to(DEV))
    assert ((got.double().cpu() - ref).norm() / ref.norm()).item() < BAR[torch.float32]
    q, k, v, par = _inputs(1, 2, 2, 9, 1, 64, torch.float32, 7)
    ln = torch.full((1, 9), 0.5)
    ref = ochord.chord_attention(q, k, v, *par, ln, 3, None)
    got = ops.apply_chord_attention(q.to(DEV), far(k), far(v), *(p.to(DEV) for p in par), ln.to(DEV), q_start=3)
    assert ((got.double().cpu() - ref).norm() / ref.norm()).item() < BAR[torch.float32]
