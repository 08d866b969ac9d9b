"""Host-side test of the shared scratch's guard: one lock per device, held by one thread at a time, and taken
again by the thread that holds it (a module that holds it calls functions that take it)."""

import threading

import pytest


def test_guard_is_one_reentrant_lock_per_device(pkg):
    S = pkg.scratch
    a = S.guard("cuda:0")
    assert S.guard("cuda:0") is a and S.guard("cuda:1") is not a
    with pytest.raises(ValueError):
        S.guard("cpu")
    order, inside = [], threading.Event()

    def other():
        inside.wait(5)
        with S.guard("cuda:0"):
            order.append("other")

    t = threading.Thread(target=other)
    t.start()
    with S.guard("cuda:0"):
        with S.guard("cuda:0"):
            inside.set()
        t.join(0.2)
        order.append("holder")
    t.join(5)
    assert order == ["holder", "other"]
