"""ops.table_choices: the experts that a table names for every token id, for all layers at once."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layers", [1, 3, 33])
@pytest.mark.parametrize("tokens", [1, 16, 300])
def test_table_choices(layers, tokens):
    from nano_vllm_x_amd import ops

    g = torch.Generator().manual_seed(layers)
    tables = [torch.randint(0, 8, (97, 1 + i % 3), generator=g, dtype=torch.int32).cuda() for i in range(layers)]
    ids = torch.randint(0, 97, (tokens,), generator=g).cuda()
    for t, (idx, wts) in zip(tables, ops.table_choices(tables, ids)):
        assert torch.equal(idx, t[ids]) and idx.is_contiguous() and wts.is_contiguous()
        assert torch.equal(wts, torch.full(idx.shape, 1.0 / t.shape[1], device="cuda"))
