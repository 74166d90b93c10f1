"""Places on a GPU that processes share (no GPU: the counting)."""
import gc
import os
import subprocess
import sys

import pytest

from nano_vllm_x_amd.core.device_places import Sharers, take_place

OTHER = "import sys; from nano_vllm_x_amd.core.device_places import take_place; p = [take_place(sys.argv[1], 2) for _ in range(3)]; print(sum(x is not None for x in p), flush=True); sys.stdin.read()"


class User:
    pass


def _other(name):
    p = subprocess.Popen([sys.executable, "-c", OTHER, name], stdin=subprocess.PIPE, stdout=subprocess.PIPE, text=True)
    return p, int(p.stdout.readline())


def _end(p):
    p.stdin.close()
    p.wait(60)
    p.stdout.close()


def test_two_places_for_all_processes():
    name = f"nvx-test-{os.getpid()}"
    mine = take_place(name, 2)
    other, got = _other(name)
    assert mine is not None and got == 1 and take_place(name, 2) is None
    _end(other)                                # (they go with their process, however it ends)
    second = take_place(name, 2)
    assert second is not None and take_place(name, 2) is None
    mine.close()
    assert take_place(name, 2).close() is None
    second.close()


@pytest.mark.parametrize("elsewhere", [0, 1, 2])
def test_more_objects_than_places_take_turns(elsewhere):
    s, dev = Sharers(f"nvx-test-{os.getpid()}-s{elsewhere}", 2, name_of=str), "gpu0"
    taken = [take_place(f"{s.name}-{dev}", 2) for _ in range(elsewhere)]
    users = []
    for n in range(1, 4):
        if not s.room(dev):
            assert elsewhere == 2              # no step goes without a place in its process
            break
        users.append(User())
        s.add(users[-1], dev)
        assert s.crowded(dev) == (n > 2 - elsewhere)
    for t in taken:
        t.close()
    if users:
        del users[0], users[0]                 # one left: one place, the others are given back
        gc.collect()
        assert not s.crowded(dev) and (other := take_place(f"{s.name}-{dev}", 2)) is not None and take_place(f"{s.name}-{dev}", 2) is None
        other.close()
        users.clear()
        gc.collect()
        both = [take_place(f"{s.name}-{dev}", 2) for _ in range(2)]
        assert all(b is not None for b in both) and not s.room(dev)
        for b in both:
            b.close()


def test_a_place_that_became_free_is_taken_for_the_next_object():
    s, dev = Sharers(f"nvx-test-{os.getpid()}-n", 2, name_of=str), "gpu0"
    other = take_place(f"{s.name}-{dev}", 2)
    users = [User(), User()]
    assert s.room(dev)
    s.add(users[0], dev)
    other.close()
    assert s.room(dev)
    s.add(users[1], dev)
    assert not s.crowded(dev)
