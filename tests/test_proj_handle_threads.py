"""A projection packed into torch's memory gets its native handle on first use (`marlin_proj._WrappingOwner`).  Threads
that use one projection for the first time together must all be given the same handle, and nobody may free it while
the projection lives.  CPU only: the library's two functions are stand-ins that hold every thread inside `wrap` until
all are there."""
import threading
from types import SimpleNamespace

import pytest
import torch

from kiln_amd import _lib, marlin_proj

THREADS = 4


@pytest.fixture
def library(monkeypatch):
    inside, lock, made, freed = threading.Barrier(THREADS), threading.Lock(), [], []

    def wrap(b, s, k, n, groupsize, dev, out):
        try:
            inside.wait(timeout=1.0)
        except threading.BrokenBarrierError:
            pass                                    # callers that come one at a time are as good
        with lock:
            made.append(0x1000 + 16 * len(made))
            out._obj.value = made[-1]
        return _lib.PROJ_OK

    monkeypatch.setattr(_lib, "load", lambda: SimpleNamespace(kiln_marlin_proj_wrap=wrap, kiln_marlin_proj_free=freed.append))
    return made, freed


def test_threads_share_one_handle_that_nobody_frees(library):
    made, freed = library
    owner = marlin_proj._WrappingOwner(torch.empty(8, 512, dtype=torch.int32), torch.empty(1, 256, dtype=torch.float16), 128, 256, 128)
    start, got = threading.Barrier(THREADS), []

    def use():
        start.wait()
        got.append(owner.handle)

    threads = [threading.Thread(target=use) for _ in range(THREADS)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=30)
    assert len(got) == THREADS and set(got) == {owner.handle}
    assert owner.handle not in freed
    assert sorted(freed + [owner.handle]) == made   # a handle that was made in vain is freed, once
    handle = owner.handle
    del owner
    assert freed.count(handle) == 1
