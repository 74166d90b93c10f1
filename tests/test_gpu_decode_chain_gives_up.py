"""Decode steps in one launch whose workgroups wait in vain: the launch ends by its clock, nothing of it passes for a result, and the runner goes on layer by layer."""
import os

import pytest
import torch

from test_gpu_decode_chain import _prefill, _runner, _sequences, _step

pytestmark = pytest.mark.gpu


def _wait_in_vain(r, monkeypatch, sizes=(1, 2, 4)):
    """From here on the graphs launch one workgroup too few: what it would leave never comes."""
    from nano_vllm_x_amd import ops

    monkeypatch.setattr(ops.DecodeChain, "SECONDS", 20e-3)
    monkeypatch.setattr(ops.DecodeChain, "WORKGROUPS", 127)
    r._capture_chain(list(sizes))
    torch.cuda.synchronize()


def _runner_with(lengths, seed=4):
    r, seqs = _runner(4, 400), _sequences(lengths, seed)
    r.initialize_kv_cache(sum(lengths) + 4 * len(lengths))
    assert r.decode_chain is not None
    _prefill(r, seqs)
    return r, seqs


def test_what_left_is_nan_and_the_next_step_says_so(monkeypatch):
    r, seqs = _runner_with((150, 7, 64))
    want = _step(r, seqs)
    _wait_in_vain(r, monkeypatch)
    for _ in range(2):                                       # a launch behind one that gave up does not wait, and ends the same way
        left = r.compute_logits(_batch(seqs))
        assert r.decode_chain is not None
    torch.cuda.synchronize()
    assert bool(left.isnan().all()) and r.decode_chain.failed
    with pytest.raises(RuntimeError, match="gave up waiting"):
        _step(r, seqs)
    assert r.decode_chain is None and r.chain_graph is None
    got, again = _step(r, seqs), _step(r, seqs)
    assert torch.equal(got, again) and float((got - want).norm() / want.norm()) < 0.02 and r.stats["chain_steps"] == 3


def _batch(seqs):
    from nano_vllm_x_amd.core.common import ForwardBatch, ForwardMode

    return ForwardBatch(forward_mode=ForwardMode.DECODE, num_seqs=len(seqs), seqs=seqs)


def _take(seqs, ids, spare):
    for s, i in zip(seqs, ids):
        s.token_ids, s.kv_indices, s.cached_kv_len = s.token_ids + [i], s.kv_indices + [spare.pop()], s.cached_kv_len + 1
        s.num_tokens += 1


def _two_steps(r, seqs, order, filters):
    """Ids of a step and of one that takes its input ids from it; `order`: launches (l) and collections (c)."""
    from nano_vllm_x_amd.core.common import SamplingParams

    for s in seqs:
        s.sampling_params = SamplingParams(temperature=0.8, top_k=20 if filters else -1)
    used, out, handles = {i for s in seqs for i in s.kv_indices}, [], []
    spare = [i for i in range(r.kv_cache_size) if i not in used]
    for what in order:
        if what == "l":
            if handles or out:
                _take(seqs, out[-1] if out else [-1] * len(seqs), spare)
            handles.append(r.launch_step(_batch(seqs), ids_on_device=list(range(len(seqs))) if len(handles) + len(out) else None))
        elif what == "w":
            torch.cuda.synchronize()
        else:
            out.append(r.finish_step(handles.pop(0)))
    return out


@pytest.mark.parametrize("filters", [False, True])
@pytest.mark.parametrize("order", ["lclc", "llcc", "lwlcc"])
@pytest.mark.parametrize("lengths", [(150, 7, 64), (90,)])
def test_steps_whose_ids_are_not_collected_are_computed_again(monkeypatch, lengths, order, filters):
    """The tokens are those of a runner that goes layer by layer, whichever step gave up and however many were on their way."""
    r, seqs = _runner_with(lengths)
    r.decode_chain = r.chain_graph = None
    want, calls = _two_steps(r, seqs, order, filters), r.sampler.calls
    r, seqs = _runner_with(lengths)
    _wait_in_vain(r, monkeypatch)
    got = _two_steps(r, seqs, order, filters)
    assert got == want and r.sampler.calls == calls and r.decode_chain is None
    assert r.stats["chain_steps_again"] == (2 if order == "llcc" else 1) and _step(r, seqs).isfinite().all()


def test_only_the_second_gives_up(monkeypatch):
    r, seqs = _runner_with((150, 7, 64))
    first = r.finish_step(r.launch_step(_with_params(seqs)))
    assert not r._chain_steps and r.stats["chain_steps"] == 1
    _wait_in_vain(r, monkeypatch)
    spare = [i for i in range(r.kv_cache_size) if i not in {i for s in seqs for i in s.kv_indices}]
    _take(seqs, [-1] * 3, spare)
    handle = r.launch_step(_batch(seqs), ids_on_device=[0, 1, 2])
    second = r.finish_step(handle)
    for s, i in zip(seqs, first):
        s.token_ids = s.token_ids[:-1] + [i]
    r.sampler.calls -= 1
    assert r.finish_step(r.launch_step(_batch(seqs))) == second and r.decode_chain is None


def _with_params(seqs):
    from nano_vllm_x_amd.core.common import SamplingParams

    for s in seqs:
        s.sampling_params = SamplingParams(temperature=0.8, top_k=-1)
    return _batch(seqs)


def test_a_step_left_uncollected_for_two_more_is_an_error(monkeypatch):
    r, seqs = _runner_with((150, 7, 64))
    _wait_in_vain(r, monkeypatch)
    handle = r.launch_step(_with_params(seqs))
    for _ in range(2):
        r.compute_logits(_batch(seqs))
    for _ in range(2):
        with pytest.raises(RuntimeError, match="cannot be computed again"):
            r.finish_step(handle)


@pytest.mark.parametrize("layers", [False, True])
def test_what_left_ahead_of_a_step_that_ended_well_is_not_told_of_later(monkeypatch, layers):
    """Whichever way that step went: a failure after it is that of another step."""
    r, seqs = _runner_with((150, 7, 64))
    _step(r, seqs)
    assert r._chain_left > 0
    graph = r.chain_graph
    if layers:
        r.chain_graph = None
    r.finish_step(r.launch_step(_with_params(seqs)))
    r.chain_graph = graph
    assert r._chain_left == 0
    _wait_in_vain(r, monkeypatch)
    r.finish_step(r.launch_step(_batch(seqs)))
    assert r.decode_chain is None and _step(r, seqs).isfinite().all()


def test_a_warm_up_that_gives_up_leaves_the_layers(monkeypatch):
    from nano_vllm_x_amd import ops

    monkeypatch.setattr(ops.DecodeChain, "SECONDS", 20e-3)
    monkeypatch.setattr(ops.DecodeChain, "WORKGROUPS", 127)
    r, seqs = _runner(1, 100), _sequences((50,), 4)
    r.initialize_kv_cache(64)
    assert r.decode_chain is None and r.chain_graph is None
    _prefill(r, seqs)
    assert _step(r, seqs).isfinite().all() and "chain_steps" not in r.stats and r.stats["graph_steps"] == 1


def test_without_a_place_or_when_asked_the_layers_are_taken(monkeypatch):
    """(Other processes of the machine hold both places of the GPU.)"""
    from nano_vllm_x_amd import ops
    from nano_vllm_x_amd.core.device_places import Sharers, device_name, take_place

    sharers = Sharers(f"nvx-test-{os.getpid()}", 2)
    monkeypatch.setattr(ops.DecodeChain, "_sharers", sharers)
    taken = [take_place(f"{sharers.name}-{device_name(0)}", 2) for _ in range(2)]
    assert all(taken)
    for _ in range(2):
        r, seqs = _runner(1, 100), _sequences((50,), 4)
        r.initialize_kv_cache(64)
        _prefill(r, seqs)
        assert r.decode_chain is None and _step(r, seqs).isfinite().all() and "chain_steps" not in r.stats
        for t in taken:
            t.close()
        monkeypatch.setenv("NVX_DECODE_CHAIN", "0")
