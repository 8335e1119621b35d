'''linear_rows refuses epilogue operands of the wrong shape or type whatever the epilogue and the
input's layout (checked on the host, before any launch).'''
import pytest
import torch

from motif.ops.linear_rows import linear_rows


@pytest.mark.parametrize('x', [torch.zeros(4, 64, dtype=torch.bfloat16), torch.zeros(4, 128, dtype=torch.bfloat16)[:, :64]], ids=['contiguous', 'strided'])
@pytest.mark.parametrize('aux', [torch.zeros(4, 31, dtype=torch.bfloat16), torch.zeros(4, 32)], ids=['shape', 'dtype'])
@pytest.mark.parametrize('name', ['aux', 'aux2'])
def test_unused_operands_are_still_checked(x, aux, name):
    with torch.no_grad(), pytest.raises(ValueError, match='epilogue operand'):
        linear_rows(x, torch.zeros(32, 64, dtype=torch.bfloat16), **{name: aux})
