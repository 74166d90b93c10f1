"""Places on a GPU that all processes of a machine share: for launches whose workgroups wait for each other and so must find room together."""
from __future__ import annotations

import socket
import threading
import weakref
from typing import Optional

import torch


def device_name(device) -> str:
    """The same in every process that sees this GPU, whatever its index there."""
    p = torch.cuda.get_device_properties(device)
    return f"{p.uuid}-{p.pci_domain_id:x}.{p.pci_bus_id:x}.{p.pci_device_id:x}"


def take_place(name: str, count: int) -> Optional[socket.socket]:
    """One of `count` places of that name, or None where others hold them all; given back when it is closed, or by the system with the process.  (The name of a socket
    without a file, which one process of a network namespace can have: nothing is left behind, no folder or owner has to agree.)"""
    for i in range(count):
        place = None
        try:
            place = socket.socket(socket.AF_UNIX, socket.SOCK_DGRAM)
            place.bind(f"\0{name}-{i}")
            return place
        except OSError:
            if place is not None:
                place.close()
    return None


class Sharers:
    """The objects of this process whose launches need one of `count` places on a GPU each.  As long as each has one they run as they like; with more objects than
    places they are `crowded` and have to follow each other."""

    def __init__(self, name: str, count: int, name_of=device_name):
        self.name, self.count, self.name_of = name, count, name_of
        self.lock = threading.RLock()       # (an object may be collected, and give its place back, inside a call that holds it)
        self._held, self._users = {}, {}

    def _count(self, device) -> int:
        return sum(1 for _ in self._users.get(device, ()))

    def room(self, device) -> bool:
        """Whether one more object may run: with a place of its own, or in turn with those that have one here."""
        with self.lock:
            held = self._held.setdefault(device, [])
            if len(held) <= self._count(device) and len(held) < self.count:
                place = take_place(f"{self.name}-{self.name_of(device)}", self.count)
                if place is not None:
                    held.append(place)
            return bool(held)

    def add(self, user, device):
        with self.lock:
            self._users.setdefault(device, weakref.WeakSet()).add(user)
        weakref.finalize(user, self._left, device).atexit = False

    def _left(self, device):
        with self.lock:
            held = self._held.get(device, [])
            while len(held) > self._count(device):
                held.pop().close()

    def crowded(self, device) -> bool:
        return self._count(device) > len(self._held.get(device, ()))
