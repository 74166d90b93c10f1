"""The state slots of a decode step travel behind its other integers."""
from types import SimpleNamespace

import torch

from nano_vllm_x_amd.layers.attention import BlockTable


def test_state_slots_go_up_with_the_step_and_padding_rows_have_none():
    bt = BlockTable(4, n_rows=9, row_capacity=8, device="cpu", with_states=True)
    assert bt.state_slots.tolist() == [-1] * 4 and int(bt.step_dev[0]) == 0
    seqs = [SimpleNamespace(seq_id=str(i), kv_indices=[3, 5 + i], token_ids=[7, 8 + i], state_slot=2 - i) for i in range(3)]
    for n in (3, 1, 2):                      # (a shorter step after a longer one: what the buffers held before is gone)
        for s in seqs[:n]:
            bt.assign(s.seq_id)
        bt.stage_decode_step(seqs[:n])
        assert bt.state_slots.tolist() == [2, 1, 0][:n] + [-1] * (4 - n)
        assert bt.step_dev[0] == n and bt.step_dev[4 + 12:4 + 12 + n].tolist() == [8, 9, 10][:n] and bt.step_dev[4 + 8:4 + 8 + n].tolist() == [5, 6, 7][:n]
    bt.clear_step()
    assert bt.state_slots.tolist() == [-1] * 4 and not bt.step_dev[:20].any()
    plain = BlockTable(4, n_rows=9, row_capacity=8, device="cpu")
    assert plain.state_slots is None and plain.step_dev.numel() == 20
