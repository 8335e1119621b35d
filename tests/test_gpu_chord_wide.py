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
