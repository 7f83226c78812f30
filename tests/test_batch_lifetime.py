"""When a Batch frees its solves (no GPU: the library calls are recorded)."""
import gc

import pytest

import minifs_amd as mfs
from minifs_amd import _lib


class RecordedCalls:
    """Stands for the library: every batch call succeeds and is counted."""

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        def call(*args):
            self.calls.append(name)
            if name == "mfs_batch_create_ex":
                args[2]._obj.value = 0x1000
            if name in ("mfs_batch_add", "mfs_batch_attach"):
                args[-1]._obj.value = self.calls.count(name) - 1
            return 0x2000 if name == "mfs_batch_ctx" else 0

        return call

    def destroyed(self):
        return self.calls.count("mfs_batch_destroy")


class AnyGrid:
    def view(self):
        return _lib.MfsMeshView()


@pytest.fixture
def calls(monkeypatch):
    gc.collect()
    gc.disable()
    rec = RecordedCalls()
    monkeypatch.setattr(mfs, "lib", lambda: rec)
    yield rec
    gc.enable()


def test_dropped_batch_is_destroyed_at_once(calls):
    b = mfs.Batch()
    members = [b.add(AnyGrid(), _lib.MfsParams()) for _ in range(3)]
    del b, members
    assert calls.destroyed() == 1


def test_member_keeps_its_batch(calls):
    b = mfs.Batch()
    m = b.add(AnyGrid(), _lib.MfsParams())
    b.add(AnyGrid(), _lib.MfsParams())
    del b
    assert calls.destroyed() == 0 and m._h
    del m
    assert calls.destroyed() == 1


def test_closed_batch_empties_its_members(calls):
    b = mfs.Batch()
    m, r = b.add(AnyGrid(), _lib.MfsParams()), b.add(AnyGrid(), _lib.MfsParams())
    b.remove(r)
    assert r._h is None and m._h and list(b.members) == [0]
    b.close()
    b.close()
    assert calls.destroyed() == 1 and m._h is None and not b.members and not b._h
    del b, m, r
    assert calls.destroyed() == 1
